// Per-subband F-stage launch.  FFT lengths 64..1024 (1024: complex) run fstage16_item
// (fstage16.hpp), a workgroup of 256 threads per group of items (station,
// FFT); longer FFTs go to fstage_big.hip.
#include "fstage16.hpp"

namespace gxc {
namespace {

using namespace fs;

// Items per workgroup of 256 threads.
constexpr int f_ipw(int L) { return 2048 / L; }

template <int L, bool CPLX, int OUT>
__global__ void __launch_bounds__((2 * (L / 16) * f_ipw(L))) __attribute__((amdgpu_waves_per_eu(8)))
fstage_kernel(FParams p) {
  __shared__ __align__(16) unsigned char smem[QLds<L, CPLX, f_ipw(L)>::BYTES];
  fstage16_item<L, CPLX, OUT, f_ipw(L)>(p, (int)xcd_order(blockIdx.x, gridDim.x), smem);
}

// Subbands of one length: units of f_ipw items, the last of a subband's partly
// empty.
template <int L, int OUT>
__global__ void __launch_bounds__((2 * (L / 16) * f_ipw(L))) __attribute__((amdgpu_waves_per_eu(8)))
fstage_group_kernel(const FSeg *__restrict__ segs, int nseg) {
  __shared__ __align__(16) unsigned char smem[QLds<L, false, f_ipw(L)>::BYTES];
  const long long u = xcd_order(blockIdx.x, gridDim.x);
  const int k = find_fseg(segs, nseg, u);
  const FParams p = segment_params(segs, k);
  fstage16_item<L, false, OUT, f_ipw(L)>(p, (int)(u - segs[k].unit0), smem);
}

template <int L>
hipError_t launch_group(const FSeg *segs, int nseg, long long units, int out_mode, hipStream_t s) {
  const dim3 grid((unsigned)units), block(2 * (L / 16) * f_ipw(L));
  switch (out_mode) {
    case OUT_F32: hipLaunchKernelGGL((fstage_group_kernel<L, OUT_F32>), grid, block, 0, s, segs, nseg); break;
    case OUT_F16: hipLaunchKernelGGL((fstage_group_kernel<L, OUT_F16>), grid, block, 0, s, segs, nseg); break;
    case OUT_BF16: hipLaunchKernelGGL((fstage_group_kernel<L, OUT_BF16>), grid, block, 0, s, segs, nseg); break;
    case OUT_FP8: hipLaunchKernelGGL((fstage_group_kernel<L, OUT_FP8>), grid, block, 0, s, segs, nseg); break;
    case OUT_POWER: hipLaunchKernelGGL((fstage_group_kernel<L, OUT_POWER>), grid, block, 0, s, segs, nseg); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <int L, bool CPLX, int OUT>
hipError_t launch_out(const FParams &p, int items, hipStream_t s) {
  constexpr int IPW = f_ipw(L);
  hipLaunchKernelGGL((fstage_kernel<L, CPLX, OUT>), dim3((unsigned)((items + IPW - 1) / IPW)),
                     dim3(2 * (L / 16) * IPW), 0, s, p);
  return hipGetLastError();
}

template <int L, bool CPLX>
hipError_t launch_one(const FParams &p, hipStream_t s) {
  const long long items = (long long)p.nant * p.nt;
  if (items <= 0) return hipSuccess;
  if (items > 0x3fffffffLL) return hipErrorInvalidValue;
  switch (p.out_mode) {
    case OUT_F32: return launch_out<L, CPLX, OUT_F32>(p, (int)items, s);
    case OUT_F16: return launch_out<L, CPLX, OUT_F16>(p, (int)items, s);
    case OUT_BF16: return launch_out<L, CPLX, OUT_BF16>(p, (int)items, s);
    case OUT_FP8: return launch_out<L, CPLX, OUT_FP8>(p, (int)items, s);
    case OUT_POWER: return launch_out<L, CPLX, OUT_POWER>(p, (int)items, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

bool fstage_supported(int L, bool cplx) {
  (void)cplx;
  return L >= 64 && L <= 32768 && (L & (L - 1)) == 0;
}

int fstage_blocks(int L, bool cplx, int *out) {
  int n = 0;
  out[n++] = L <= 4096 ? 256 : L == 8192 ? 512 : L / 32;
  if (L <= 2048) out[n++] = 128;
  if (L <= 4096 && L >= (cplx ? 256 : 128)) out[n++] = 512;
  if (L >= 2048 && L <= 8192) out[n++] = L / 32;
  return n;
}

namespace {

hipError_t launch_piece(const FParams &p, int L, bool cplx, hipStream_t s) {
  if (f_matrix(L)) return launch_fstage_big(p, L, cplx, s);
  if (fstage_one_wave(L, !cplx)) return launch_fstage_1k(p, s);
#define GXC_F_CASE(LL) \
  case LL: return cplx ? launch_one<LL, true>(p, s) : launch_one<LL, false>(p, s);
  switch (L) {
    GXC_F_CASE(64)
    GXC_F_CASE(128)
    GXC_F_CASE(256)
    GXC_F_CASE(512)
    case 1024: return launch_one<1024, true>(p, s);
    default: return hipErrorInvalidValue;
  }
#undef GXC_F_CASE
}

}  // namespace

long long fstage_units(int L, long long items) {
  const int ipw = L < 1024 ? f_ipw(L) : 1;
  return (items + ipw - 1) / ipw;
}

hipError_t launch_fstage_group(const FSeg *segs, int nseg, long long units, int L, int out_mode, hipStream_t s) {
  if (units <= 0) return hipSuccess;
  if (units > 0x7fffffffLL) return hipErrorInvalidValue;
  switch (L) {
    case 256: return launch_group<256>(segs, nseg, units, out_mode, s);
    case 512: return launch_group<512>(segs, nseg, units, out_mode, s);
    case 1024: return launch_fstage_1k_group(segs, nseg, units, out_mode, s);
    default: return launch_fstage_big_group(segs, nseg, units, L, out_mode, s);
  }
}

int fstage_most_ffts(int L, int nant) {
  const long long n = 0xff000000LL / ((long long)nant * (L / 8));
  return (int)(n < 1 ? 1 : n > 0x7fffffff ? 0x7fffffff : n);
}

hipError_t launch_fstage(const FParams &p, int L, bool cplx, int block, hipStream_t s) {
  if (block == kFBlockMfma)
    return fstage_mfma_supported(L, cplx, p.out_mode == OUT_F32) ? launch_fstage_mfma(p, L, s) : hipErrorInvalidValue;
  const int most = fstage_most_ffts(L, p.nant);
  FParams q = p;
  for (int t = 0; t < p.nt || t == 0; t += q.nt) {
    const size_t bin = (size_t)t * p.nant * 2 * (cplx ? L : L / 2);  // of the piece's first FFT
    q.t0 = p.t0 + t * p.tstride;
    q.nt = p.nt - t < most ? p.nt - t : most;
    if (t > 0) {
      if (p.out_mode == OUT_F32)
        q.spectra = p.spectra + bin;
      else if (p.out_mode == OUT_POWER)
        q.power = p.power + bin;
      else
        q.out = static_cast<unsigned char *>(p.out) + bin * (p.out_mode == OUT_FP8 ? 2 : 4);
    }
    const hipError_t e = launch_piece(q, L, cplx, s);
    if (e != hipSuccess || q.nt <= 0) return e;
  }
  return hipSuccess;
}

}  // namespace gxc
