// The F-stage of 1024 real points: one wave per (station, FFT), radices 32 * 32.
// Pass 0 of both polarisations runs on the matrix cores (fstage_pass0.hpp): the
// wave's 64 lanes hold 32 columns of 16 outputs each per polarisation.  One
// exchange through LDS, a component at a time, then lanes 0..31 run the last
// pass of polarisation A and lanes 32..63 that of B, 32 points each, of which
// the 16 kept bins leave as runs of 32 neighbours.  No barriers, and one
// exchange where the 16-point form (fstage16.hpp) has two and does the unpacking,
// rotation and first pass on the VALU: 5 stations x 20000 FFTs 0.295 -> 0.264 ms.
// What bounds it is VALU issue at 4 waves per SIMD (114 registers), half of it
// the delay split, tables and matrix of the item; the split by one wave for
// four in a workgroup was slower (0.280 ms).  Complex input stays with the
// 16-point form, which writes and reads at the rate of HBM.
#pragma once

#include "fstage_pass0.hpp"

namespace gxc {
namespace fs {
namespace one {

constexpr int L = 1024, T = 32, NCHAN = 512, kTables = f_tw_size(L);
using TG = TabGeom<L, false>;
static_assert(T % TG::S2 == 0 && 16 % TG::S == 0, "table offsets");

// LDS of a wave: two planes of 1024 words (before the exchange the operands of
// M), the tables, the level pairs and the packed samples.
constexpr int kTab = 8 * L, kLut = kTab + TG::NTAB * 8, kStage = kLut + 128, kBytes = kStage + L / 2;
static_assert(MatLds<false>::BYTES <= 8 * L, "M's operands fit the planes");

// Item = station + nant * FFT; smem holds kBytes bytes, 16-byte aligned.
template <int OUT>
__device__ __forceinline__ void fstage_1k_item(const FParams &p, int item, unsigned char *smem) {
  float2 *sub = reinterpret_cast<float2 *>(smem + kTab), *step = sub + TG::S2;
  float2 *fsub = step + TG::NSTEPS, *fstep = fsub + TG::S;
  uint2 *slut = reinterpret_cast<uint2 *>(smem + kLut);
  uint32_t *stage = reinterpret_cast<uint32_t *>(smem + kStage);
  float *plane = reinterpret_cast<float *>(smem);
  const int lane = threadIdx.x;
  const int tl = item / p.nant, st = item - tl * p.nant, t = p.t0 + tl * p.tstride;
  constexpr unsigned EB = out_bytes(OUT);
  unsigned char *out = out_base<OUT>(p) + (size_t)item * 2 * (NCHAN * EB);
  double frac, a, b;
  int offset;
  const bool ok = split_offset<L>(p, st, t, offset, frac, a, b);
  offset = __builtin_amdgcn_readfirstlane(offset);
  const bool valid = __builtin_amdgcn_readfirstlane(ok ? 1 : 0) != 0;
  if (lane == 0 && OUT != OUT_POWER) p.valid[(size_t)st * p.numffts + t] = valid ? 1 : 0;
  if (!valid) {
    for (unsigned q = lane; q < 2 * NCHAN; q += 64) store_val<OUT>(out + q * EB, make_float2(0.f, 0.f), 1.f);
    return;
  }
  const float2 *tw = p.twiddle + kTables;
  Pass0In<L, false, true, 2> in;
  in.template load<64>((gbyte *)p.station[st], offset, lane, lane);
  fill_tables<L, false>(p, frac, a, b, sub, lane, 64, pass0_unscale<false>());
  if (lane < 16) slut[lane] = level_pair(lane);
  in.template put<64>(stage, lane);
  __syncthreads();
  build_matrix<false, 64>(smem, step, T / TG::S2, tw, lane);
  __syncthreads();
  const int c = lane & 15, g = lane >> 4, j0 = 2 * c;
  floatx4 acc[2][2][2][2];  // [polarisation][column][row half][component]
  in.fetch(stage, lane);
#pragma unroll
  for (int pol = 0; pol < 2; pol++) {
    in.matmul(acc[pol], smem, slut, pol);
    // one step after the other: mixed they spill 20 registers (0.305 ms)
    __builtin_amdgcn_sched_barrier(0);
    finish_columns<L, false, 2>(acc[pol], sub, step, tw, j0, g);
    __builtin_amdgcn_sched_barrier(0);
  }
  __syncthreads();  // M's operands are read
  // point 32 jj + r of a plane: rows of 8 chunks of 4 at chunk position
  // (r / 4) ^ (jj / 2 mod 8): eight neighbouring lanes of a store, and the 32
  // lanes of a load, cover the 32 banks once
  float2 v[32];
  const int r = lane & 31;
  const float *from = plane + (lane >> 5) * L + (r & 3);
#pragma unroll
  for (int comp = 0; comp < 2; comp++) {
#pragma unroll
    for (int pol = 0; pol < 2; pol++)
#pragma unroll
      for (int e = 0; e < 2; e++)
#pragma unroll
        for (int rh = 0; rh < 2; rh++)
          *reinterpret_cast<floatx4 *>(plane + pol * L + 32 * (j0 + e) + 4 * ((g ^ (c & 7)) ^ (4 * rh))) =
              acc[pol][e][rh][comp];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 32; k++) {
      const float x = from[32 * k + 4 * ((r >> 2) ^ ((k >> 1) & 7))];
      if (comp)
        v[k].y = x;
      else
        v[k].x = x;
    }
    __syncthreads();
  }
  __builtin_amdgcn_sched_barrier(0);
  dft<32>(v);
  __builtin_amdgcn_sched_barrier(0);
  // bins q = r + 32 k < nchan times the fractional-sample rotator
  // (fxkernel.cpp:614-625); q / S = r / S + a compile-time step
  const int pol = lane >> 5;
  unsigned char *row = out + (unsigned)pol * (NCHAN * EB);
  const float2 f0 = fsub[r % TG::S];
#pragma unroll
  for (int k = 0; k < 16; k++) {
    const unsigned q = r + 32 * k;
    const float2 y = cmul(cmul(f0, fstep[r / TG::S + k * (32 / TG::S)]), v[k]);
    store_val<OUT>(row + q * EB, y, bin_scale<OUT, NCHAN>(p, 2 * st + pol, q));
  }
}

}  // namespace one
}  // namespace fs
}  // namespace gxc
