// Internal declarations shared by the HIP kernels and the C-ABI host code.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace gxc {

constexpr double kPi = 3.14159265358979323846;  // IPP_PI (fxkernel/src/vectordefs.h:8)
constexpr float kHiMag = 3.3359f;                // fxkernel/src/fxkernel.cpp:17

constexpr int ilog2c(int x) { return x <= 1 ? 0 : 1 + ilog2c(x / 2); }

// Geometry shared by the host and the F-stage kernel for FFT length L.
// Generalised stride: s = 2^floor(log2(nchan)/2) (fxkernel.cpp:58-64 only
// accepts square nchan, for which this is sqrt(nchan)).
struct Geometry {
  int L, nchan, s, S2, nsteps, fracsteps;
  static Geometry make(int nchan, bool cplx) {
    Geometry g{};
    g.nchan = nchan;
    g.L = cplx ? nchan : 2 * nchan;
    g.s = 1 << (ilog2c(nchan) / 2);
    g.S2 = cplx ? g.s : 2 * g.s;
    g.nsteps = g.L / g.S2;
    g.fracsteps = nchan / g.s;
    return g;
  }
};

// FFT passes of the F-stage at length L: radix of pass p (1: no such pass),
// product of the radices before it, number of passes.  From 2048 points on
// pass 0 is a radix-32 pass on the matrix cores and a thread holds 32 points
// (fstage_big.hpp), below 16 (fstage16.hpp).
constexpr bool f_matrix(int L) { return L >= 2048; }
constexpr int f_radix(int L, int p) {
  return p == 0   ? (f_matrix(L) ? 32 : 16)
         : p == 1 ? (f_matrix(L) ? 32 : L == 256 ? 16 : L == 64 ? 4 : 8)
                  : L / (f_radix(L, 0) * f_radix(L, 1));
}
constexpr int f_ns(int L, int p) { return p == 0 ? 1 : f_ns(L, p - 1) * f_radix(L, p - 1); }
constexpr int f_npass(int L) { return f_radix(L, 2) == 1 ? 2 : 3; }
// Twiddle tables of one FFT length, in float2 entries:
//   W_32^m (m < 32);
//   matrix pass 0: W_1024^(k1 r), applied to its outputs r < 32 for pass-1
//   input k1 < 32: [r / 16][r / 2 % 2][r / 4 % 4][k1][r % 2]; and for the last
//   pass of radix R, [power][m] W_L^(power m) of every second m < 1024 (every
//   m at radix 32): a thread loads its first butterfly's powers and takes
//   constants on top for the others;
//   VALU passes of radix R after NS points: [power][m < NS] W_(NS R)^(power m);
// for the powers 1, 2, 3, 4, 8, .. R/2.  Neighbouring lanes read neighbouring
// entries: gathers from one table of W_L, up to a 128-byte line per lane, kept
// the vector L1 busy 64 % of the F-stage (16 stations x 4096 channels).
constexpr int f_npowers(int R) { return R == 2 ? 1 : R == 4 ? 3 : 2 + ilog2c(R) - 1; }
constexpr int f_power(int i) { return i < 3 ? i + 1 : 4 << (i - 3); }
constexpr int f_tw_first(int L) { return f_matrix(L) ? 2 : 1; }  // first pass with a power table
constexpr int f_tw_step(int L, int p) { return !f_matrix(L) || f_radix(L, p) >= 32 ? 1 : 2; }
constexpr int f_tw_entries(int L, int p) { return f_ns(L, p) / f_tw_step(L, p); }
constexpr int f_tw_off(int L, int p) {
  return p == f_tw_first(L) ? 32 + (f_matrix(L) ? 1024 : 0)
                            : f_tw_off(L, p - 1) + f_npowers(f_radix(L, p - 1)) * f_tw_entries(L, p - 1);
}
constexpr int f_tw_size(int L) { return f_tw_off(L, f_npass(L)); }
// Real input of 1024 points: a wave per (station, FFT), radices 32 * 32
// (fstage_1k.hpp); its W_32 and W_1024 follow the length's other tables.
constexpr bool fstage_one_wave(int L, bool real) { return L == 1024 && real; }

// What the F-stage writes per (station, FFT): FP32 spectra, scaled
// reduced-precision spectra (complex: 2 x 16 bits or 2 x 8 bits), or |X|^2
// accumulated per (input, channel) for the scale estimate.
enum OutMode { OUT_F32 = 0, OUT_F16 = 1, OUT_BF16 = 2, OUT_FP8 = 3, OUT_POWER = 4 };

// Arguments of the F-stage kernel (unpack, fringe rotate, FFT, fractional
// sample correction) for FFTs t0 + i*tstride, i in [0, nt), of every station.
struct FParams {
  const uint8_t *const *station;  // [nant] device pointers to packed input
  const double *delays;           // [nant][4]: d0, d1, d2, file offset (s)
  const float *subchanfreq;       // [s]          fxkernel.cpp:173
  const float *stepchanfreq;      // [fracsteps]  fxkernel.cpp:174
  const float2 *twiddle;          // [f_tw_size(L)]
  float2 *spectra;                // OUT_F32: [nt][nant*2][nchan]
  void *out;                      // OUT_F16/BF16/FP8: [nt][nant*2][nchan] packed complex
  const float *scales;            // [nant*2][nchan] multipliers before rounding
  float *power;                   // OUT_POWER: [nt][nant*2][nchan] |X|^2 per sampled FFT
  uint8_t *valid;                 // [nant][numffts]
  // Missing VDIF frames (nullptr: none): frame_ok[st][f] != 0 when frame f,
  // samples [f, f+1) * frame_samples[st], is present; an FFT touching a
  // missing frame is invalid for that station.
  const uint8_t *const *frame_ok;
  const int *frame_samples;
  int out_mode;
  int t0, nt, tstride, nant, numffts;
  int maxoffset;                  // (numffts-1)*L
  int stepmul;                    // s (stride law) or S2 (exact phase)
  int fraclo;                     // LO has a fractional part
  double lo, lofrac, sampletime;
  double samplerate;              // 1 / sampletime
};

// Row counts: for each output row (station pair; autos have j == k) the
// number of FFTs in which both stations were valid.
struct CountParams {
  const uint8_t *valid;  // [nant][numffts]
  const int2 *rowmap;    // [nrows]
  int *counts;           // [nrows]
  int *host_counts;      // the same in pinned host memory, or null
  int numffts, nrows;
};

// One subband's share of a multi-subband launch (units of segment k are
// unit0[k] .. unit0[k+1]-1, segments in increasing unit0).
struct FSeg {  // units = fstage_units
  FParams p;
  long long unit0;
  int L;
};
struct CountSeg {  // units = nrows
  CountParams p;
  long long unit0;
};

// Workgroups that keep every CU busy for a persistent launch of `kernel`
// (occupancy x CU count), at most `total`.
long long persistent_grid(const void *kernel, int block, size_t dyn_lds, long long total);

// Allow `kernel` dynamic LDS of `bytes` (above the 64 KiB default) on the
// current device, once per (device, kernel, bytes); safe from any thread.
hipError_t allow_dynamic_lds(const void *kernel, int bytes);

// Launchers (defined in the .hip files).  Return hipSuccess or the launch error.
bool fstage_supported(int L, bool cplx);
// Values that gxc_config.fblock may have at FFT length L (default first): the
// workgroup sizes of earlier kernels, which a tuning run may have written down.
// They all run the length's one kernel, whose workgroup has 64 threads at 1024
// real points, 256 at other lengths below 2048 and L/32 from there on.
int fstage_blocks(int L, bool cplx, int *out /* [4] */);
// FFTs of nant stations that one launch takes at length L: a grid has fewer
// than 2^32 work items, and the kernels at most L/8 per (station, FFT).  From
// 2^32 on (32 stations x 64 points: 16.7 million FFTs) launch_fstage launches in
// pieces.
int fstage_most_ffts(int L, int nant);
// block: kFBlockMfma, else one of fstage_blocks (0 = default), which all run
// the length's one kernel
hipError_t launch_fstage(const FParams &p, int L, bool cplx, int block, hipStream_t s);
hipError_t launch_fstage_big(const FParams &p, int L, bool cplx, hipStream_t s);  // L = 2048..32768
hipError_t launch_fstage_1k(const FParams &p, hipStream_t s);                     // L = 1024, real
// The F-stage of several subbands of one length in one launch, real input, L =
// 256..8192.  Its work items, L/8 at most per (station, FFT), have to stay
// below 2^32 (fstage_most_ffts).
long long fstage_units(int L, long long items);
hipError_t launch_fstage_group(const FSeg *segs, int nseg, long long units, int L, int out_mode, hipStream_t s);
hipError_t launch_fstage_big_group(const FSeg *segs, int nseg, long long units, int L, int out_mode, hipStream_t s);
hipError_t launch_fstage_1k_group(const FSeg *segs, int nseg, long long units, int out_mode, hipStream_t s);
// Subbands of several of these lengths in one launch, longest first
// (fstage_mixed.hip): taken up to kFMixedUnits units per launch that it saves.
constexpr int kFMixedUnits = 1500;
hipError_t launch_fstage_mixed(const FSeg *segs, int nseg, long long units, int out_mode, hipStream_t s);
// F-stage with the FFT passes on the matrix cores (fstage_mfma.hip): real
// input; reduced-precision outputs (and the power pass) at L = 2048..8192,
// FP32 spectra (operands as f16 hi + lo) at L = 2048..4096.
constexpr int kFBlockMfma = -1;
bool fstage_mfma_supported(int L, bool cplx, bool fp32);
hipError_t launch_fstage_mfma(const FParams &p, int L, hipStream_t s);
hipError_t launch_counts(const CountParams &p, hipStream_t s);
hipError_t launch_counts_multi(const CountSeg *segs, int nseg, long long total, hipStream_t s);

}  // namespace gxc
