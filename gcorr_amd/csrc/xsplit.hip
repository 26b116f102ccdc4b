// Streaming X-stage: FP16 and BF16 spectra of up to 32 inputs, and the F-stage's
// FP32 spectra, on the 16-bit matrix cores.
//
// FP32: every value x is taken as hi + lo, two f16 (x - hi is exact and has at
// most 13 bits, of which lo keeps 11 and its sign: 2^-24 of x, an FP32
// rounding), and every product x y as hi hi + hi lo + lo hi with FP32 sums.  The
// term left out, lo lo, is 2^-24 of the product and of random sign, except
// where an input meets itself: the blocks on the diagonal take it as well.
//
// For channel c over FFTs t, with x_a = a_a + i b_a (a = input index):
//   Re V_ab = sum_t a_a a_b + b_a b_b,  Im V_ab = sum_t b_a a_b - a_a b_b
// so with K slots (a, b) of 16 FFTs one v_mfma_f32_16x16x32_f16 of the slots
// [a, b] with [a, b] adds to Re, and one with [-b, a] to Im.  A 16-bit complex
// value is such a slot pair as it lies in memory.
//
// The FP32 spectra come from the framework's own F-stage, whose |X| is at most L
// times the largest sample: p.scale, a power of two, brings that below f16's
// largest value.  f16 rounds a lo part to 2^-25 at least, whatever its size.
// 2-bit spectra are of rms sqrt(L) and more, scaled 54 and more, and lose
// nothing by it.  Complex ones are of rms 1 where a window holds one sample of
// one level: the loss is then 2^-25 / scale, and from 4096 points on (scale
// below kLiftBelow) lo parts are kept times 2^6 (LIFT), so that it is 2^-24 at
// 32768 points.  A K-step's products with lo parts are taken down before they
// join; where sums run on (64 inputs), the hi parts that meet lo parts are.
// Errors of such visibilities against 64 bits with FP32 products, without LIFT
// and with it: 2048 points 6.0e-7, 2.7e-7, -; 8192 points (10 stations) 8.0e-7,
// 1.7e-6, 3.6e-7; 32768 points (8 stations) 8.8e-7, 7.6e-6, 4.1e-7.  X-stage in
// the same order: 8 x 32768 x 1000 FFTs 0.78, 0.65, 0.66 ms; 12 x 16384 x 800
// 0.68, 0.48, 0.54; 32 x 4096 x 1500 1.22, 0.61, 0.70.
// Spectra handed in by a caller have no such bound and take xengine.hip's FP32
// products.
//
// What bounds it is the reading of the spectra: the FP32 matrix products that
// it replaces kept the MFMAs busy for 70 % of the time, here they, the VALU
// (the split: about 20 instructions per value and wave) and LDS are busy for
// 15-30 %.  A workgroup takes 32 channels (FP32, 33 and more inputs: 16; 16-bit:
// 64) of all M inputs, so that a row is 256 bytes (with 128 the same kernel read
// 5.5 instead of 6.2 TB/s; a plain read of this pattern reaches 5.5-6.2 and
// 6.4).  Stages of SB FFTs go straight from memory to LDS in 16-byte units into
// a ring of five, four of them under way; the lanes of a row take its units in
// an order rotated by the row, so that the 16 lanes of an operand read find 16
// distinct bank groups (at 16 and 32 inputs; at 12 half of the LDS's cycles are
// conflicts, 7 % of all).  A wave owns the channels of one unit (33 and more
// inputs: one channel), so each value is read from LDS and split once.
// Nontemporal loads, since a row is read once: 3.21 -> 2.94 ms at 16 stations
// before the ring.
// X-stage, before -> with this, FP32: 16 stations x 4096 channels x 15625 FFTs
// 3.18 -> 2.64 ms (6.2 TB/s), 6 x 1024 x 62500 1.16 -> 0.93 ms, 32 x 1024 x 6000
// 1.15 -> 0.63 ms, a batch of 8 subbands x 8 stations 3.45 -> 2.47 ms.  Errors of
// the visibilities against 64 bits (with the F-stage's): 3.6e-7 -> 1.4e-7, 5.1e-7
// -> 1.6e-7, 4.5e-7 -> 4.0e-7, 9.5e-7 -> 3.3e-7.  16-bit (loads through registers,
// one stage ahead, 8 or 16 FFTs transposed per lane): 16 x 4096 x 15625 1.46 ->
// 1.41 ms, 10 x 2048 x 5001 0.217 -> 0.143 ms, 8 x 32768 x 1000 0.460 -> 0.367 ms.
#include <algorithm>
#include <cmath>

#include "xengine_common.hpp"

namespace gxc {
namespace {

using namespace xs;

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kNontemporal = 2;                               // cache policy of a load
constexpr int kVmcnt(int n) { return 0x0f70 | (n & 15); }  // s_waitcnt vmcnt(n), n < 16


template <int ET, int MB>
struct XS {
  static constexpr bool F32 = ET == OUT_F32;
  static constexpr int CB = F32 ? 8 : 4;           // bytes of a complex value
  static constexpr int CT = F32 ? (MB == 4 ? 16 : 32) : 64;  // channels of a workgroup
  static constexpr int CPW = F32 ? (MB == 4 ? 1 : 2) : 4;    // channels per wave
  static constexpr int NWV = CT / CPW, NTHR = 64 * NWV;
  static constexpr int ROWB = CT * CB;
  static constexpr int UPR = ROWB / 16, RPI = 64 / UPR;  // 16-byte units per row, rows per load instruction
  // unit u of a row lies at position u ^ swz(row)
  __device__ static constexpr int swz(int row) { return UPR == 8 ? (row >> 1) & 7 : row & 15; }
  static constexpr int SB = MB == 1 ? 8 : 4;   // FFTs per stage
  static constexpr int NU = SB / 4;            // a lane's units of an input and stage
  // FFTs per MFMA: 16 (K = 32), or 8 (K = 16) where the 96 running sums of four
  // channels leave no registers for the operands of 16
  static constexpr int KF = !F32 && MB == 2 ? 8 : 16, KD = KF / 4;
  static constexpr int NST = KF / SB;          // stages per MFMA K-step
  static constexpr int RING = 5;               // stages in LDS: 160 KiB at 16, 32 and 64 inputs
  static constexpr int NTILE = MB * (MB + 1) / 2;
  // the stages' rows, and those that padded inputs of the last FFT read
  static int lds_bytes(int M) { return ROWB * (RING * SB * M + 16 * MB - M); }
};

// An MFMA operand of one lane: KD pairs (a, b), one per FFT.
template <int KD>
struct Op {
  uint32_t d[KD];
};
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short short4v __attribute__((ext_vector_type(4)));
template <int ET>
__device__ __forceinline__ floatx4 mfma(const Op<4> &a, const Op<4> &b, floatx4 c) {
  if constexpr (ET == OUT_BF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                    0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0, 0,
                                                   0);
}
template <int ET>
__device__ __forceinline__ floatx4 mfma(const Op<2> &a, const Op<2> &b, floatx4 c) {
  if constexpr (ET == OUT_BF16)
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(short4v, a), __builtin_bit_cast(short4v, b), c,
                                                     0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(half4, a), __builtin_bit_cast(half4, b), c, 0, 0,
                                                 0);
}

// (re, im) * scale as an f16 pair and the f16 pair of the remainder (LIFT: times
// kLift; at most half a unit of f16's largest values, 16, so 2^10)
constexpr float kLift = 64.f, kUnlift = 1.f / kLift;
constexpr float kLiftBelow = 0.125f;  // p.scale; real input has 0.5 and more
template <bool LIFT>
__device__ __forceinline__ void split(float re, float im, float scale, uint32_t &hi, uint32_t &lo) {
  const floatx2 x = {re * scale, im * scale};
  const half2v h = __builtin_convertvector(x, half2v);
  const floatx2 b = __builtin_convertvector(h, floatx2);
  floatx2 d = {x.x - b.x, x.y - b.y};
  if constexpr (LIFT) d = {d.x * kLift, d.y * kLift};
  hi = __builtin_bit_cast(uint32_t, h);
  lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(d, half2v));
}

// an operand of hi parts for a product with lifted lo parts (and lo parts taken
// down)
template <int KD>
__device__ __forceinline__ Op<KD> unlift(const Op<KD> &v) {
  Op<KD> w;
#pragma unroll
  for (int i = 0; i < KD; i++)
    w.d[i] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2v, v.d[i]) * (half2v){(_Float16)kUnlift, (_Float16)kUnlift});
  return w;
}

// [a, b] -> [-b, a]
template <int KD>
__device__ __forceinline__ Op<KD> turn(const Op<KD> &v) {
  Op<KD> w;
#pragma unroll
  for (int i = 0; i < KD; i++) w.d[i] = __builtin_amdgcn_alignbit(v.d[i], v.d[i], 16) ^ 0x00008000u;
  return w;
}

typedef __attribute__((address_space(1))) void gvoid;
typedef __attribute__((address_space(3))) void lvoid;

// Two 16-byte (or four 8-byte) operand units from LDS, waited for: in a block
// of its own the compiler does not wait for the loads to LDS that are under
// way.
__device__ __forceinline__ void read_units(floatx4 &a, floatx4 &b, unsigned addr0, unsigned addr1) {
  asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %3\n\ts_waitcnt lgkmcnt(0)"
               : "=&v"(a), "=&v"(b)
               : "v"(addr0), "v"(addr1)
               : "memory");
}
__device__ __forceinline__ void read_blocks(floatx4 &a, floatx4 &b, unsigned addr) {
  asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %2 offset:%3\n\ts_waitcnt lgkmcnt(0)"
               : "=&v"(a), "=&v"(b)
               : "v"(addr), "n"(16 * 256)
               : "memory");
}
__device__ __forceinline__ void read_blocks(floatx2 &a, floatx2 &b, floatx2 &c, floatx2 &d, unsigned addr) {
  asm volatile(
      "ds_read_b64 %0, %4\n\tds_read_b64 %1, %4 offset:2048\n\tds_read_b64 %2, %4 offset:4096\n\t"
      "ds_read_b64 %3, %4 offset:6144\n\ts_waitcnt lgkmcnt(0)"
      : "=&v"(a), "=&v"(b), "=&v"(c), "=&v"(d)
      : "v"(addr)
      : "memory");
}

// Channels CT group .., FFT split `unit_split`, on a workgroup of XS::NTHR
// threads (every thread calls it with the same arguments: it contains
// barriers).  lds holds XS::lds_bytes(M) bytes, 16-byte aligned.
template <int ET, int MB, bool LIFT = false>
__device__ __forceinline__ void xsplit_item(const XMParams &p, int group_, int unit_split, unsigned char *lds) {
  const int group = __builtin_amdgcn_readfirstlane(group_), split_ = __builtin_amdgcn_readfirstlane(unit_split);
  using X = XS<ET, MB>;
  static_assert(X::F32 || !LIFT, "lo parts");
  constexpr int CPW = X::CPW, SB = X::SB, KD = X::KD;
  static_assert(X::F32 || X::ROWB == 256, "read_blocks");
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int M = p.M, l15 = lane & 15, g = lane >> 4;
  // uniform, which 64-bit divisions on the VALU hide
  const int tb = __builtin_amdgcn_readfirstlane((int)((long long)p.nt * split_ / p.splits));
  const int te = __builtin_amdgcn_readfirstlane((int)((long long)p.nt * (split_ + 1) / p.splits));
  const size_t rowbytes = (size_t)p.nchan * X::CB;
  const unsigned char *src = static_cast<const unsigned char *>(p.spectra) + (size_t)group * X::ROWB;
  const int stage_bytes = SB * M * X::ROWB;

  // A wave's load instruction fills 64 units, RPI rows (row = t M + input) of
  // a stage; it has nld, at most two, per stage, NWV RPI rows apart (a multiple
  // of 16: the same rotation).  Rows at and past te read the last one.
  const int lrow = X::RPI * wave + lane / X::UPR, pairq = (lane % X::UPR) ^ X::swz(lrow);
  const int nld = (SB * M / X::RPI - wave + X::NWV - 1) / X::NWV;
  auto request = [&](int ts, int slot) {
    const int t = ts < te ? ts : te - 1, last = (te - t < SB ? te - t : SB) * M - 1;
    const unsigned char *base = src + (size_t)t * M * rowbytes;
    unsigned char *d = lds + slot * stage_bytes + 1024 * wave;
#pragma unroll
    for (int k = 0; k < 2; k++) {
      const int row = lrow + X::RPI * k * X::NWV;
      // rowbytes < 2^24 (xsplit_channels), so at most 127 rows fit 31 bits
      const unsigned off = __umul24(row < last ? row : last, (unsigned)rowbytes) + 16u * pairq;
      if (k < nld)
        __builtin_amdgcn_global_load_lds((gvoid *)(base + off), (lvoid *)(d + 1024 * k * X::NWV), 16, 0, kNontemporal);
    }
  };

  // operand reads: FFT 4 u + g of a stage, input 16 b + l15.  (Lanes of
  // inputs past M read other rows: what they make of them lands in rows and
  // columns past M.)
  const int pw = CPW == 1 ? wave >> 1 : wave;
  unsigned addr[X::NU];
#pragma unroll
  for (int u = 0; u < X::NU; u++) {
    const int row = (4 * u + g) * M + l15;
    addr[u] = (unsigned)(uintptr_t)(lvoid *)lds + row * X::ROWB + 16 * (pw ^ X::swz(row)) +
              (CPW == 1 ? 8 * (wave & 1) : 0);
  }

  floatx4 re[CPW][X::NTILE], im[CPW][X::NTILE];
#pragma unroll
  for (int c = 0; c < CPW; c++)
#pragma unroll
    for (int t = 0; t < X::NTILE; t++) re[c][t] = im[c][t] = floatx4{0, 0, 0, 0};

  const int nst = tb < te ? (te - tb + X::KF - 1) / X::KF * X::NST : 0;  // stages
  for (int n = 0; n < X::RING - 1 && n < nst; n++) request(tb + n * SB, n);
  int slot = 0;
  for (int n0 = 0; n0 < nst; n0 += X::NST) {
    typedef float unit __attribute__((ext_vector_type(CPW == 1 ? 2 : 4)));
    Op<KD> H[CPW][MB], L[CPW][MB];  // K slots: FFTs 4 i + g in d[i]; L: FP32 only
#pragma unroll
    for (int s = 0; s < X::NST; s++) {
      const int n = n0 + s;
      // this wave's loads of stage n have arrived: those of the RING - 2
      // stages after it may be under way
      if (n + X::RING - 2 >= nst || nld == 0)
        __builtin_amdgcn_s_waitcnt(kVmcnt(0));
      else if (nld == 1)
        __builtin_amdgcn_s_waitcnt(kVmcnt(X::RING - 2));
      else
        __builtin_amdgcn_s_waitcnt(kVmcnt(2 * (X::RING - 2)));
      // every wave's have, and stage n - 1 is read (a barrier without the fence
      // that would wait for every load)
      __builtin_amdgcn_s_barrier();
      if (n + X::RING - 1 < nst) request(tb + (n + X::RING - 1) * SB, slot == 0 ? X::RING - 1 : slot - 1);
      const unsigned so = slot * stage_bytes;
      unit raw[MB][X::NU];
      if constexpr (MB == 1)
        read_units(raw[0][0], raw[0][1], addr[0] + so, addr[1] + so);
      else if constexpr (MB == 2)
        read_blocks(raw[0][0], raw[1][0], addr[0] + so);
      else
        read_blocks(raw[0][0], raw[1][0], raw[2][0], raw[3][0], addr[0] + so);
      slot = slot + 1 == X::RING ? 0 : slot + 1;
#pragma unroll
      for (int u = 0; u < X::NU; u++) {
        if (tb + (n + 1) * SB > te) {
          const bool in = tb + n * SB + 4 * u + g < te;
#pragma unroll
          for (int b = 0; b < MB; b++) raw[b][u] = in ? raw[b][u] : (unit)0.f;
        }
#pragma unroll
        for (int c = 0; c < CPW; c++)
#pragma unroll
          for (int b = 0; b < MB; b++) {
            uint32_t &h = H[c][b].d[s * X::NU + u];
            if constexpr (X::F32)
              split<LIFT>(raw[b][u][2 * c], raw[b][u][2 * c + 1], p.scale, h, L[c][b].d[s * X::NU + u]);
            else
              h = __builtin_bit_cast(uint32_t, (float)raw[b][u][c]);
          }
      }
    }
#pragma unroll
    for (int c = 0; c < CPW; c++) {
#pragma unroll
      for (int bj = 0; bj < MB; bj++) {
        // The products of one kind for all blocks of a column, then the next:
        // two MFMAs on one sum are MB others apart.  FP32, up to 32 inputs: a
        // K-step's products are summed by themselves, small ones first, and
        // added once (one rounding of the running sum instead of four); at 64
        // inputs the registers hold only the running sums.
        constexpr bool OWN = X::F32 && MB <= 2;
        floatx4 *sr = re[c] + bj * (bj + 1) / 2, *sq = im[c] + bj * (bj + 1) / 2;
        floatx4 r[MB], q[MB];
#pragma unroll
        for (int bi = 0; bi <= bj; bi++) {
          r[bi] = OWN ? floatx4{0, 0, 0, 0} : sr[bi];
          q[bi] = OWN ? floatx4{0, 0, 0, 0} : sq[bi];
        }
        if constexpr (X::F32) {
          // LIFT: a K-step's own sums are taken down before the hi products
          // join; running sums take lifted lo parts times hi parts taken down
          constexpr bool DOWN = LIFT && !OWN;
          const Op<KD> l = DOWN ? unlift(L[c][bj]) : L[c][bj];
          r[bj] = mfma<ET>(l, l, r[bj]);
          if constexpr (LIFT && OWN) r[bj] *= kUnlift;
          const Op<KD> w = turn(L[c][bj]);
#pragma unroll
          for (int bi = 0; bi <= bj; bi++) {
            const Op<KD> h = DOWN ? unlift(H[c][bi]) : H[c][bi];
            r[bi] = mfma<ET>(h, L[c][bj], r[bi]);
            q[bi] = mfma<ET>(h, w, q[bi]);
          }
          const Op<KD> h = DOWN ? unlift(H[c][bj]) : H[c][bj], wh = turn(h);
#pragma unroll
          for (int bi = 0; bi <= bj; bi++) {
            r[bi] = mfma<ET>(L[c][bi], h, r[bi]);
            q[bi] = mfma<ET>(L[c][bi], wh, q[bi]);
          }
          if constexpr (LIFT && OWN)
#pragma unroll
            for (int bi = 0; bi <= bj; bi++) r[bi] *= kUnlift, q[bi] *= kUnlift;
        }
        const Op<KD> w = turn(H[c][bj]);
#pragma unroll
        for (int bi = 0; bi <= bj; bi++) {
          r[bi] = mfma<ET>(H[c][bi], H[c][bj], r[bi]);
          q[bi] = mfma<ET>(H[c][bi], w, q[bi]);
        }
#pragma unroll
        for (int bi = 0; bi <= bj; bi++) {
          sr[bi] = OWN ? sr[bi] + r[bi] : r[bi];
          sq[bi] = OWN ? sq[bi] + q[bi] : q[bi];
        }
        if constexpr (MB == 4) __builtin_amdgcn_sched_barrier(0);
      }
    }
  }

  // D[i][j] of a 16x16 tile sits in lane j + 16*(i/4), element i%4.  Blocks on
  // the diagonal hold Im V in both triangles: half of each, so that the
  // finalise's difference gives Im V back.
  const size_t MM = (size_t)M * M;
  int zero = 0;
  asm volatile("" : "+s"(zero));  // the lane is worked out here, not held over the loop
  const int tid = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, zero));
  const float us = X::F32 ? p.unscale : 1.f, ush = 0.5f * us;
#pragma unroll
  for (int c = 0; c < CPW; c++) {
    const int ch = group * X::CT + wave * CPW + c;
    const size_t off = ((size_t)split_ * p.nchan + ch) * 2 * MM;
    float *pre = p.partial + off, *pim = pre + MM;
    float *cre = p.comp ? p.comp + off : nullptr, *cim = p.comp ? cre + MM : nullptr;
    int tile = 0;
#pragma unroll
    for (int bj = 0; bj < MB; bj++)
#pragma unroll
      for (int bi = 0; bi <= bj; bi++, tile++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int a = 16 * bi + 4 * (tid >> 4) + r, b = 16 * bj + (tid & 15);
          if (a < M && b < M) {
            const size_t ab = (size_t)a * M + b, ba = (size_t)b * M + a;
            put_partial(p.accumulate, pre, cre, ab, re[c][tile][r] * us);
            put_partial(p.accumulate, pim, cim, ab, im[c][tile][r] * (bi == bj ? ush : us));
            if (bi != bj) put_partial(p.accumulate, pim, cim, ba, 0.f);
          }
        }
  }
}

template <int ET, int MB, bool LIFT>
__global__ void __launch_bounds__((XS<ET, MB>::NTHR)) __attribute__((amdgpu_waves_per_eu(4))) xsplit_kernel(XMParams p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int groups = p.nchan / XS<ET, MB>::CT;
  const long long u = xcd_swizzle(blockIdx.x, (long long)groups * p.splits);
  xsplit_item<ET, MB, LIFT>(p, (int)(u % groups), (int)(u / groups), lds);
}

// Several subbands of the same M: unit = (subband, split, channel group), a
// workgroup each.
template <int ET, int MB>
__global__ void __launch_bounds__((XS<ET, MB>::NTHR)) __attribute__((amdgpu_waves_per_eu(4)))
xsplit_multi_kernel(const XSeg *__restrict__ segs, int nseg) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const long long u = xcd_swizzle(blockIdx.x, gridDim.x);
  const int k = __builtin_amdgcn_readfirstlane(find_seg(segs, nseg, u));
  const XMParams p = segs[k].p;
  const int local = (int)(u - segs[k].unit0), groups = p.nchan / XS<ET, MB>::CT;
  xsplit_item<ET, MB>(p, local % groups, local / groups, lds);
}

template <int ET, int MB, bool LIFT>
hipError_t launch_lift(const XMParams &p, hipStream_t s) {
  using X = XS<ET, MB>;
  const long long units = (long long)(p.nchan / X::CT) * p.splits;
  if (p.nchan % X::CT || units > 0x7fffffffLL) return hipErrorInvalidValue;
  const hipError_t e =
      allow_dynamic_lds(reinterpret_cast<const void *>(&xsplit_kernel<ET, MB, LIFT>), X::lds_bytes(16 * MB));
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((xsplit_kernel<ET, MB, LIFT>), dim3((unsigned)units), dim3(X::NTHR), X::lds_bytes(p.M), s, p);
  return hipGetLastError();
}
template <int ET, int MB>
hipError_t launch_mb(const XMParams &p, hipStream_t s) {
  if constexpr (ET == OUT_F32)
    if (p.scale < kLiftBelow) return launch_lift<ET, MB, true>(p, s);
  return launch_lift<ET, MB, false>(p, s);
}

template <int ET, int MB>
hipError_t launch_multi_mb(const XSeg *segs, int nseg, long long total, int M, hipStream_t s) {
  using X = XS<ET, MB>;
  const void *fn = reinterpret_cast<const void *>(&xsplit_multi_kernel<ET, MB>);
  const hipError_t e = allow_dynamic_lds(fn, X::lds_bytes(16 * MB));
  if (e != hipSuccess) return e;
  if (total > 0x7fffffffLL) return hipErrorInvalidValue;
  hipLaunchKernelGGL((xsplit_multi_kernel<ET, MB>), dim3((unsigned)total), dim3(X::NTHR), X::lds_bytes(M), s, segs,
                     nseg);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_xsplit(const XMParams &p, int out_mode, hipStream_t s) {
  const int mb = xm_blocks(p.M);
  switch (out_mode * 8 + mb) {
    case OUT_F32 * 8 + 1: return launch_mb<OUT_F32, 1>(p, s);
    case OUT_F32 * 8 + 2: return launch_mb<OUT_F32, 2>(p, s);
    case OUT_F32 * 8 + 4: return launch_mb<OUT_F32, 4>(p, s);
    case OUT_F16 * 8 + 1: return launch_mb<OUT_F16, 1>(p, s);
    case OUT_F16 * 8 + 2: return launch_mb<OUT_F16, 2>(p, s);
    case OUT_BF16 * 8 + 1: return launch_mb<OUT_BF16, 1>(p, s);
    case OUT_BF16 * 8 + 2: return launch_mb<OUT_BF16, 2>(p, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_xsplit_multi(const XSeg *segs, int nseg, long long total, int out_mode, int M, hipStream_t s) {
  if (total <= 0) return hipSuccess;
  switch (out_mode * 8 + xm_blocks(M)) {
    case OUT_F32 * 8 + 1: return launch_multi_mb<OUT_F32, 1>(segs, nseg, total, M, s);
    case OUT_F32 * 8 + 2: return launch_multi_mb<OUT_F32, 2>(segs, nseg, total, M, s);
    case OUT_F32 * 8 + 4: return launch_multi_mb<OUT_F32, 4>(segs, nseg, total, M, s);
    case OUT_F16 * 8 + 1: return launch_multi_mb<OUT_F16, 1>(segs, nseg, total, M, s);
    case OUT_F16 * 8 + 2: return launch_multi_mb<OUT_F16, 2>(segs, nseg, total, M, s);
    case OUT_BF16 * 8 + 1: return launch_multi_mb<OUT_BF16, 1>(segs, nseg, total, M, s);
    case OUT_BF16 * 8 + 2: return launch_multi_mb<OUT_BF16, 2>(segs, nseg, total, M, s);
    default: return hipErrorInvalidValue;
  }
}

int xsplit_channels(int out_mode, int M, int nchan) {
  const int ct = out_mode == OUT_F32                        ? (M > 32 ? 16 : 32)
                 : out_mode == OUT_F16 || out_mode == OUT_BF16 ? (M > 32 ? 0 : 64)
                                                               : 0;
  // request()'s 24-bit products: rows of 2^24 bytes (2^22 channels of 16 bits,
  // which a caller's spectra may have) and more go through xengine.hip
  const bool fits = (long long)nchan * (out_mode == OUT_F32 ? 8 : 4) < 1 << 24;
  return ct && nchan % ct == 0 && fits ? ct : 0;
}

// The general kernel has four to eight times the workgroups, each with a quarter
// to an eighth of the channels, and wins where these cannot fill the chip and a
// CU's own bandwidth binds.  At up to 16 inputs it wins nowhere.  X-stage and
// finalise, general against streaming: FP32, 20 inputs, 2048 channels, 100 FFTs (33
// MB of spectra) 37 : 41 us, 200 FFTs (66 MB) 56 : 49; 512 channels, 400 FFTs (33
// MB) 40 : 43, 800 FFTs 51 : 49; 32 inputs, 512 x 400 (52 MB) 51 : 52, 512 x 800
// 71 : 63; FP16, 32 inputs, 512 x 800 (52 MB) 51 : 58, 512 x 1600 76 : 73; 64 inputs,
// FP32, 512 x 100 (26 MB) 67 : 70, 512 x 200 (52 MB) 91 : 74.  With 256 groups of
// channels the chip is full at any length: 32 inputs, 8192 x 20 FP32 70 : 63.
bool xsplit_better(int out_mode, int M, int nchan, int nt) {
  const int ct = xsplit_channels(out_mode, M, nchan), mb = xm_blocks(M);
  if (!ct || mb == 1) return ct != 0;
  const double bytes = (double)nt * M * nchan * xm_element_bytes(out_mode);
  return nchan / ct >= 256 || bytes >= (mb == 2 ? 56 << 20 : 32 << 20);
}

// One workgroup per CU, which its LDS admits at 16, 32 and 64 inputs, where
// there are FFTs enough: 6 stations x 1024 channels 0.93 ms with 256
// workgroups, 0.96 with 512; 16 x 4096 2.59 with 256, 2.64 with 1024.  Short
// subintegrations have fewer splits:
//   a split saves its share of the loop and adds to the finalise's, ~M/9 FFTs'
//   time each: the two meet at 3 sqrt(nt / M) splits;
//   with many channels the writing and reading of the partials adds more, 8 M^2
//   bytes per channel at ~3 TB/s: they meet at 25 sqrt(nt / (nchan sqrt M));
//   16 FFTs, a K-step, at least;
//   4 at a time, which the finalise has in flight together, and one rather than
//   two unless they are long (its copy of one split is quicker).
// FP32, whole pass in us with 1, 2, 4, 8, 16, 64 splits, the choice in brackets: 30
// stations x 256 channels x 500 FFTs 209, 159, 120, [114], 150; 8 x 512 x 200 58, 51,
// 46, [44], 46; 24 x 1024 x 100 [91], 93, 86, 107; 3 x 32 x 5000 467, 255, 147, 91, 63,
// [48], 256: 61.
int xsplit_choose_splits(int out_mode, int M, int nchan, int nt) {
  const long long groups = nchan / std::max(1, xsplit_channels(out_mode, M, nchan));
  const double finalise = 3 * std::sqrt((double)nt / M);
  const double partials = 25 * std::sqrt(nt / (nchan * std::sqrt((double)M)));
  const double most = std::min({256.0, finalise, partials, nt / 16.0});
  const int s = (int)std::max(1.0, std::min<double>((256 + groups - 1) / groups, most));
  if (s >= 3) return (s + 1) / 4 * 4;
  return s == 2 && nt < 4LL * M ? 1 : s;
}

// the largest |X| of an F-stage of L points is L times the largest sample
float xsplit_scale(int L, bool cplx) {
  const double peak = (double)L * (cplx ? 128.0 * 1.4142135623730951 : (double)kHiMag);
  return (float)std::exp2(std::floor(std::log2(65000.0 / peak)));
}

}  // namespace gxc
