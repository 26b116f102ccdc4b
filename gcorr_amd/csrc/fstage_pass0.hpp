// First pass of the F-stage: packed samples to the outputs of one radix-32
// pass on the matrix cores (FFT lengths of 2048 and more, and 1024 real points)
// or of one radix-16 pass on the VALU, and the twiddles of the later passes.
#pragma once

#include "fstage_common.hpp"

namespace gxc {
namespace fs {

// v[k] *= w^k for k = 1 .. R-1, w = W_(NS R)^m (times_powers<R, 0>).  Only w^1 .. w^3 and
// w^(4 * 2^i) come from the pass's table; w^(4a) is the product of the loaded
// powers of the bits of a and w^(4a + b) = w^(4a) w^b, at most three FP32
// products (a few ulps) from table entries: four FP32 instructions of one
// wave cost less than a load's lines in the L1 that four SIMDs share.
struct Powers {
  float2 p1, p2, p3, q0, q1, q2;  // w, w^2, w^3, w^4, w^8, w^16
};
template <int A>
__device__ __forceinline__ float2 power4(const Powers &w) {  // w^(4 A)
  if constexpr (A == 1) return w.q0;
  if constexpr (A == 2) return w.q1;
  if constexpr (A == 3) return cmul(w.q0, w.q1);
  if constexpr (A == 4) return w.q2;
  if constexpr (A == 5) return cmul(w.q0, w.q2);
  if constexpr (A == 6) return cmul(w.q1, w.q2);
  return cmul(cmul(w.q0, w.q1), w.q2);
}
template <int R, int A>
__device__ __forceinline__ void times_powers(float2 *v, const Powers &w) {
  if constexpr (A == 0) {
    v[1] = cmul(v[1], w.p1);
    v[2] = cmul(v[2], w.p2);
    v[3] = cmul(v[3], w.p3);
  } else if constexpr (4 * A < R) {
    const float2 w4 = power4<A>(w);
    v[4 * A] = cmul(v[4 * A], w4);
    v[4 * A + 1] = cmul(v[4 * A + 1], cmul(w4, w.p1));
    v[4 * A + 2] = cmul(v[4 * A + 2], cmul(w4, w.p2));
    v[4 * A + 3] = cmul(v[4 * A + 3], cmul(w4, w.p3));
  }
  if constexpr (4 * A + 4 < R) times_powers<R, A + 1>(v, w);
}
template <int R, int NS, int OFF>
__device__ __forceinline__ Powers load_powers(const float2 *__restrict__ tw, unsigned m) {
  // 32-bit byte offsets from the table's uniform base
  const unsigned char *twb = reinterpret_cast<const unsigned char *>(tw + OFF);
  auto ld = [&](unsigned i) { return *reinterpret_cast<const float2 *>(twb + (8u * m + 8u * NS * i)); };
  Powers w;
  w.p1 = ld(0);
  w.p2 = w.p3 = w.q0 = w.q1 = w.q2 = w.p1;
  if constexpr (R > 2) w.p2 = ld(1), w.p3 = ld(2);
  if constexpr (R > 4) w.q0 = ld(3);
  if constexpr (R > 8) w.q1 = ld(4);
  if constexpr (R > 16) w.q2 = ld(5);
  return w;
}

// ---- pass 0 on the matrix cores ----------------------------------------
//
// Window sample n = j + k*T (T = L/32 columns j, k < 32) carries the rotator
// sub[n % S2] * step[n / S2] (fxkernel.cpp:553-558).  S2 divides T and step[]
// is a geometric sequence, so it is rho_j * E_k with rho_j = sub[j % S2] *
// step[j / S2] and E_k = step[k * T/S2], and the first radix-32 pass is
//   Y[r][j] = rho_j * sum_k M[r][k] x[j + k*T],   M[r][k] = W_32^(rk) E_k:
// a matrix product whose right-hand side is the bare samples.  Those are
// small numbers that f16 holds exactly (complex 8-bit: integers; 2-bit: +-1
// and +-3.3359f, the latter as 3.3359375 plus a remainder), so only M is
// split, into f16 hi + lo (22 bits), and the sums are FP32.  M depends on the
// (station, FFT) alone and serves its two polarisations; rows r + 16 are
// rows r with the odd k negated, so 16 rows are built and kept.  The radix-32
// butterflies, half the rotator product and most of the unpacking leave the
// VALU.
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ floatx4 mfma16(const uint4 &a, const uint4 &b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0, 0,
                                                0);
}

// (x, y) as an f16 pair and the f16 pair of the remainder
__device__ __forceinline__ void split_f16(float x, float y, uint32_t &hi, uint32_t &lo) {
  const half2v h = __builtin_convertvector((floatx2){x, y}, half2v);
  const floatx2 b = __builtin_convertvector(h, floatx2);
  hi = __builtin_bit_cast(uint32_t, h);
  lo = __builtin_bit_cast(uint32_t, __builtin_convertvector((floatx2){x - b.x, y - b.y}, half2v));
}

// Scales (powers of two) that keep the f16 remainders in the normal range:
// of the 2-bit levels and of M.  The fractional-sample factors of the last
// pass divide them out.
constexpr float kLevScale = 64.f, kMatScale = 4.f;
template <bool CPLX>
constexpr float pass0_unscale() { return CPLX ? 1.f / kMatScale : 1.f / (kMatScale * kLevScale); }

// f16 pairs of the 2-bit levels of two samples, by the 4-bit index code0 |
// code1 << 2 (fxkernel.cpp:15-28): .x the levels, .y their remainders.
__device__ __forceinline__ uint2 level_pair(int idx) {
  const float l0 = (idx & 1) == ((idx >> 1) & 1) ? kHiMag : 1.0f;
  const float l1 = ((idx >> 2) & 1) == ((idx >> 3) & 1) ? kHiMag : 1.0f;
  uint2 v;
  split_f16(kLevScale * ((idx & 2) ? l0 : -l0), kLevScale * ((idx & 8) ? l1 : -l1), v.x, v.y);
  return v;
}

// Operands of M for one (station, FFT) in LDS: 16-byte A operands of
// v_mfma_f32_16x16x32_f16, [component][hi, lo][K-step][lane], K = the 32
// samples (real) or (re, im) of 16 samples per K-step (complex, K-step ks
// holding samples 16 ks ..).  Threads 0 .. 127 (or 63 twice) build 4 samples
// of one row each.
template <bool CPLX>
struct MatLds {
  static constexpr int KS = CPLX ? 2 : 1;
  static constexpr int BYTES = 2 * 2 * KS * 1024;
};

// (estep: entries of step[] between samples k and k + 1, i.e. L/32 / S2.)
template <bool CPLX, int NTHR>
__device__ __forceinline__ void build_matrix(unsigned char *mat, const float2 *step, int estep,
                                             const float2 *__restrict__ w32, int tid) {
  constexpr int KS = MatLds<CPLX>::KS;
  for (int q = tid; q < 128; q += NTHR) {
    // neighbouring threads: the two halves of one 16-byte operand (real)
    const int kq = CPLX ? q >> 4 : (q & 1) | ((q >> 5) << 1), r = CPLX ? q & 15 : (q >> 1) & 15;
    float2 m[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int k = 4 * kq + i;
      const float2 e = step[k * estep], w = w32[(r * k) & 31];
      m[i] = cmul(w, make_float2(e.x * kMatScale, e.y * kMatScale));
    }
    if constexpr (!CPLX) {
      uint2 v[2][2];  // [component][hi, lo]
      split_f16(m[0].x, m[1].x, v[0][0].x, v[0][1].x);
      split_f16(m[2].x, m[3].x, v[0][0].y, v[0][1].y);
      split_f16(m[0].y, m[1].y, v[1][0].x, v[1][1].x);
      split_f16(m[2].y, m[3].y, v[1][0].y, v[1][1].y);
      unsigned char *d = mat + 16 * (r + 16 * (kq >> 1)) + 8 * (kq & 1);
#pragma unroll
      for (int ch = 0; ch < 4; ch++) *reinterpret_cast<uint2 *>(d + ch * 1024) = v[ch >> 1][ch & 1];
    } else {
      // (re, im) columns: real part [re, -im], imaginary part [im, re]
      uint32_t rh[4], rl[4], ih[4], il[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        split_f16(m[i].x, -m[i].y, rh[i], rl[i]);
        split_f16(m[i].y, m[i].x, ih[i], il[i]);
      }
      unsigned char *d = mat + (kq >> 2) * 1024 + 16 * (r + 16 * (kq & 3));
      *reinterpret_cast<uint4 *>(d) = make_uint4(rh[0], rh[1], rh[2], rh[3]);
      *reinterpret_cast<uint4 *>(d + KS * 1024) = make_uint4(rl[0], rl[1], rl[2], rl[3]);
      *reinterpret_cast<uint4 *>(d + 2 * KS * 1024) = make_uint4(ih[0], ih[1], ih[2], ih[3]);
      *reinterpret_cast<uint4 *>(d + 3 * KS * 1024) = make_uint4(il[0], il[1], il[2], il[3]);
    }
  }
}

// rows r + 16 of an operand of M: the odd samples negated
template <bool CPLX>
__device__ __forceinline__ uint4 upper_rows(uint4 a) {
  if constexpr (CPLX)
    return make_uint4(a.x, a.y ^ 0x80008000u, a.z, a.w ^ 0x80008000u);
  else
    return make_uint4(a.x ^ 0x80000000u, a.y ^ 0x80000000u, a.z ^ 0x80000000u, a.w ^ 0x80000000u);
}

// Input and product of one lane of a wave that holds 16 NT columns: lane
// (c, g) of the wave's 64 has columns j0 + e, j0 = NT (16 w + c), in tiles e <
// NT, and their samples k = 8 g .. 8 g + 7 (real) or k = 16 ks + 4 g + 0..3
// (complex).
//   Real: the item's L/2 bytes (both polarisations) go through LDS, loaded as
// aligned 32-bit words by neighbouring threads and shifted so that word d
// holds window samples 8 d .. 8 d + 7; a lane then reads the byte or half
// word with its NT samples.  (Loaded per lane, at byte addresses, the samples
// alone took 40 cycles of the vector L1 per load.)  The window's last word
// reaches into the next one: the buffer holds a whole FFT past the last
// window (fxkernel/src/common.cpp:16).
//   Complex: a lane loads the NT neighbouring words [Are, Aim, Bre, Bim].
template <int L, bool CPLX, bool MF, int NT>
struct Pass0In {
  static constexpr int T = L / 32, KS = MatLds<CPLX>::KS;
  static_assert(NT == 2 || NT == 4, "samples of one load");
  static constexpr int NW = CPLX ? 8 * NT : 8;
  uint32_t raw[NW];
  int sh;

  // jt: thread of the NTHR of the item; j: thread of its polarisation
  template <int NTHR>
  __device__ __forceinline__ void load(gbyte *src, int offset, int j, int jt) {
    if constexpr (CPLX) {
      const int c = j & 15, g = (j >> 4) & 3, s0 = offset + 16 * NT * (j >> 6) + NT * c;
      typedef uint32_t words __attribute__((ext_vector_type(NT), aligned(4)));
      gbyte *b0 = src + 4 * ((size_t)s0 + (size_t)(4 * g) * T);
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const words w = *reinterpret_cast<const __attribute__((address_space(1))) words *>(
            b0 + (size_t)4 * (16 * (i >> 2) + (i & 3)) * T);
#pragma unroll
        for (int e = 0; e < NT; e++) raw[NT * i + e] = w[e];
      }
    } else {
      static_assert((L / 8) % NTHR == 0 && 2 * (L / 8 / NTHR) <= NW, "whole words per thread");
      const uintptr_t a = (uintptr_t)(src + (offset >> 1));
      const __attribute__((address_space(1))) uint32_t *w =
          (const __attribute__((address_space(1))) uint32_t *)(a & ~(uintptr_t)3) + jt;
      sh = 8 * (int)(a & 3) + 4 * (offset & 1);
#pragma unroll
      for (int i = 0; i < L / 8 / NTHR; i++) {
        raw[2 * i] = w[i * NTHR];
        raw[2 * i + 1] = w[i * NTHR + 1];
      }
    }
  }
  template <int NTHR>
  __device__ __forceinline__ void put(uint32_t *stage, int jt) const {
    if constexpr (!CPLX)
#pragma unroll
      for (int i = 0; i < L / 8 / NTHR; i++)
        stage[jt + i * NTHR] = __builtin_amdgcn_alignbit(raw[2 * i + 1], raw[2 * i], (unsigned)sh);
  }
  // after a barrier
  __device__ __forceinline__ void fetch(const uint32_t *stage, int j) {
    if constexpr (!CPLX) {
      const unsigned char *b = reinterpret_cast<const unsigned char *>(stage) +
                               (16 * NT * (j >> 6) + NT * (j & 15)) / 2 + 4 * T * ((j >> 4) & 3);
#pragma unroll
      for (int i = 0; i < 8; i++)
        raw[i] = NT == 2 ? (uint32_t)b[i * (T / 2)] : (uint32_t) * reinterpret_cast<const uint16_t *>(b + i * (T / 2));
    }
  }

  // acc[tile][row half][component]: rows r = 16 rh + 4 g + i of column j0 +
  // tile; M's operands from LDS, or (one K-step) from registers
  __device__ __forceinline__ void matmul(floatx4 (&acc)[NT][2][2], const unsigned char *smat, const uint2 *slut,
                                         int pol) {
    product(acc, slut, pol, [&](int comp, int hl, int ks) {
      return reinterpret_cast<const uint4 *>(smat)[((comp * 2 + hl) * KS + ks) * 64 + (threadIdx.x & 63)];
    });
  }
  __device__ __forceinline__ void matmul(floatx4 (&acc)[NT][2][2], const uint4 (&am)[2][2], const uint2 *slut, int pol) {
    static_assert(KS == 1, "2-bit input");
    product(acc, slut, pol, [&](int comp, int hl, int) { return am[comp][hl]; });
  }

 private:
  template <typename Operand>
  __device__ __forceinline__ void product(floatx4 (&acc)[NT][2][2], const uint2 *slut, int pol, Operand operand) {
    // B operands: [tile][K-step], for 2-bit input also the remainders
    uint32_t bh[NT][KS][4], bl[NT][4];
    if constexpr (CPLX) {
      // bytes to f16: 1024 + (v + 128) has v + 128 in its low mantissa bits
      const uint32_t sel = pol ? 0x04030402u : 0x04010400u;
#pragma unroll
      for (int i = 0; i < 8; i++)
#pragma unroll
        for (int e = 0; e < NT; e++) {
          const uint32_t v = __builtin_amdgcn_perm(0x64646464u, raw[NT * i + e] ^ 0x80808080u, sel);
          const half2v h = __builtin_bit_cast(half2v, v) + (half2v){(_Float16)-1152.f, (_Float16)-1152.f};
          bh[e][i >> 2][i & 3] = __builtin_bit_cast(uint32_t, h);
        }
    } else {
#pragma unroll
      for (int i = 0; i < 4; i++) {
        // nibble e: the codes of samples k and k + 1 of column j0 + e
        const uint32_t x = raw[2 * i] >> (2 * pol), y = raw[2 * i + 1] >> (2 * pol);
        const uint32_t n = (x & 0x3333u) | ((y & 0x3333u) << 2);
#pragma unroll
        for (int e = 0; e < NT; e++) {
          const uint2 v = slut[(n >> (4 * e)) & 15u];
          bh[e][0][i] = v.x;
          bl[e][i] = v.y;
        }
      }
    }
#pragma unroll
    for (int comp = 0; comp < 2; comp++)
#pragma unroll
      for (int ks = 0; ks < KS; ks++) {
        uint4 ah = operand(comp, 0, ks), al = operand(comp, 1, ks);
#pragma unroll
        for (int rh = 0; rh < 2; rh++) {
          if (rh) ah = upper_rows<CPLX>(ah), al = upper_rows<CPLX>(al);
#pragma unroll
          for (int e = 0; e < NT; e++) {
            const uint4 xh = make_uint4(bh[e][ks][0], bh[e][ks][1], bh[e][ks][2], bh[e][ks][3]);
            floatx4 y = ks ? acc[e][rh][comp] : floatx4{0.f, 0.f, 0.f, 0.f};
            if constexpr (!CPLX) y = mfma16(ah, make_uint4(bl[e][0], bl[e][1], bl[e][2], bl[e][3]), y);
            y = mfma16(al, xh, y);
            acc[e][rh][comp] = mfma16(ah, xh, y);
          }
        }
      }
  }
};

// rho_j of column j = TR k1 + b (TR = L/1024, b < TR) is sub[TR k1 % S2]
// step[TR k1 / S2] times the rotator's turn over b samples.  Pass 1 runs over
// k1 at one b, so the first factor joins pass 1's twiddle W_1024^(r k1), once
// for the columns of a k1, and the second, kIncs[i] samples' turn, joins the
// powers of the last pass's twiddle, which runs over b: one product per point
// instead of two (8192 points, 16 stations: F-stage 5.98 -> 5.80 ms; 32768 complex
// 1.43 -> 1.34 ms).  At 2048 points (TR = 2) a thread's four columns have two k1:
// less is saved and 15 registers spill (6 stations: 2.26 -> 2.43 ms), so there
// each column takes its whole rho.
template <int L>
constexpr bool rho_in_passes() { return L >= 4096; }
constexpr int kNumIncs = 6;
__device__ __forceinline__ int inc_samples(int i) { return i < 3 ? i + 1 : 4 << (i - 3); }  // 1, 2, 3, 4, 8, 16
__device__ __forceinline__ float2 inc_entry(const FParams &p, double a, double over_l, int i) {
#pragma clang fp contract(off)
  const double ph = -((double)inc_samples(i) * over_l * a * p.lo);
  float sn, cs;
  sincospif((float)(2.0 * (ph - rint(ph))), &sn, &cs);
  return make_float2(cs, sn);
}
template <int L>
__device__ __forceinline__ Powers turn_powers(Powers w, const float2 *inc) {
  constexpr int R = L / 1024;
  if constexpr (!rho_in_passes<L>()) return w;
  w.p1 = cmul(w.p1, inc[0]);
  if constexpr (R > 2) w.p2 = cmul(w.p2, inc[1]), w.p3 = cmul(w.p3, inc[2]);
  if constexpr (R > 4) w.q0 = cmul(w.q0, inc[3]);
  if constexpr (R > 8) w.q1 = cmul(w.q1, inc[4]);
  if constexpr (R > 16) w.q2 = cmul(w.q2, inc[5]);
  return w;
}

// Outputs r of columns j0 + e times W_1024^(r k1) and rho (its first factor).
template <int L, bool CPLX, int NT>
__device__ __forceinline__ void finish_columns(floatx4 (&acc)[NT][2][2], const float2 *sub, const float2 *step,
                                               const float2 *__restrict__ tw, int j0, int g) {
  constexpr int S2 = TabGeom<L, CPLX>::S2, TR = L / 1024;
  constexpr bool IN_PASSES = rho_in_passes<L>();
  static_assert(S2 % TR == 0, "rho's factors");
  const unsigned char *wb = reinterpret_cast<const unsigned char *>(tw + 32);
  float2 pw[8];
#pragma unroll
  for (int e = 0; e < NT; e++) {
    if (e % TR == 0) {
      const unsigned k1 = (unsigned)(j0 + e) / TR;
#pragma unroll
      for (int i = 0; i < 4; i++) {  // rows 16 (i / 2) + 4 g + 2 (i % 2) + 0, 1
        const float4 w = *reinterpret_cast<const float4 *>(wb + (16u * (32u * (unsigned)g + k1) + 2048u * i));
        pw[2 * i] = make_float2(w.x, w.y);
        pw[2 * i + 1] = make_float2(w.z, w.w);
      }
      if constexpr (IN_PASSES) {
        const float2 rho = cmul(sub[k1 * TR % S2], step[k1 * TR / S2]);
#pragma unroll
        for (int i = 0; i < 8; i++) pw[i] = cmul(rho, pw[i]);
      }
    }
    float2 rho;
    if constexpr (!IN_PASSES) rho = cmul(sub[(j0 + e) % S2], step[(j0 + e) / S2]);
#pragma unroll
    for (int i = 0; i < 8; i++) {
      float2 y = make_float2(acc[e][i >> 2][0][i & 3], acc[e][i >> 2][1][i & 3]);
      if constexpr (!IN_PASSES) y = cmul(y, rho);
      const float2 x = cmul(y, pw[i]);
      acc[e][i >> 2][0][i & 3] = x.x;
      acc[e][i >> 2][1][i & 3] = x.y;
    }
  }
}

// ---- pass 0 on the VALU ----------------------------------------------------
// Thread j of L/16 has samples n = j + k*L/16, k < 16.
template <int L, bool CPLX, int NT>
struct Pass0In<L, CPLX, false, NT> {
  static constexpr int T = L / 16;
  uint32_t raw[16];
  int sh;

  __device__ __forceinline__ void load(gbyte *src, int offset, int j) {
    // T is even, so every k shares the byte parity of offset + j
    const int s0 = offset + j;
    sh = (s0 & 1) * 4;
    gbyte *b0 = src + (CPLX ? 4 * (size_t)s0 : (size_t)(s0 >> 1));
#pragma unroll
    for (int k = 0; k < 16; k++)
      raw[k] = CPLX ? *reinterpret_cast<const __attribute__((address_space(1))) uint32_t *>(b0 + (size_t)4 * k * T)
                    : (uint32_t)b0[(size_t)k * (T / 2)];
  }

  // rotator sub[n % S2] * step[n / S2] (fxkernel.cpp:553-558) times the sample
  __device__ __forceinline__ void rotate(float2 (&v)[16], const float2 *sub, const float2 *step, const float *lut,
                                         int pol, int j) const {
    constexpr int S2 = TabGeom<L, CPLX>::S2;
    const int b = CPLX ? 16 * pol : sh + 2 * pol;
#pragma unroll
    for (int k = 0; k < 16; k++) {
      const int n = j + k * T;
      const float2 r = cmul(sub[n % S2], step[n / S2]);
      if constexpr (CPLX) {
        const uint32_t w = raw[k] >> b;
        v[k] = cmul(r, make_float2((float)(int8_t)(w & 0xff), (float)(int8_t)((w >> 8) & 0xff)));
      } else {
        const float x = lut[(raw[k] >> b) & 3u];
        v[k] = make_float2(x * r.x, x * r.y);
      }
    }
  }
};

}  // namespace fs
}  // namespace gxc
