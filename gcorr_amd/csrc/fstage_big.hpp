// The F-stage for FFT lengths 2048..32768 as a device function over one
// (station, FFT) with its polarisations in turn (real input up to 8192
// points) or one (station, FFT, polarisation):
//   - L/32 threads, 32 points per thread: pass 0 (radix 32) on the matrix cores
//     (fstage_pass0.hpp), pass 1 (radix 32) and the last pass on the VALU;
//   - between passes the points go through LDS one component plane at a time
//     (L words, no padding), which the samples and the matrix operands use
//     before.
// Small workgroups with a plane each keep four waves per SIMD from four and
// more independent workgroups: forms with 16 points per thread and twice the
// waves, with both polarisations side by side, and with a pipeline over items
// in a persistent workgroup all measured 3-15 % slower at 8192 points (their
// waves met at barriers more often and wrote as much LDS).
// What bounds it: VALU issue (45 instructions per point, ~2.7 cycles each: 4 of
// the 5.8 ms below) and LDS writes (~80 bytes per clock and CU: 2 ms), which 16
// waves per CU overlap in part.  16 stations x 4096 channels x 15625 FFTs (FP32,
// 16.4 GB of spectra): 6.7 ms with the first pass on the VALU and both
// polarisations in registers, 5.8 ms now; 6 stations x 1024 channels 3.3 -> 2.26
// ms, 10 stations x 2048 channels (BF16) 1.05 -> 0.49 ms.
#pragma once

#include "fstage_pass0.hpp"

namespace gxc {
namespace fs {

// CON_: most neighbouring butterflies of the last pass per thread
template <int L, bool CPLX, int CON_ = 2>
struct BG {
  using TG = TabGeom<L, CPLX>;
  static constexpr int T = L / 32;  // threads, 32 points each
  static constexpr int RL = L / 1024;            // radix of the last pass
  static constexpr int NB = 32 / RL;             // its butterflies per thread,
  static constexpr int CON = NB < CON_ ? NB : CON_;  // CON neighbouring ones
  static constexpr int GRP = NB / CON;           // in each of GRP groups
  static constexpr int KEEP = CPLX ? RL : RL / 2;  // outputs kept per butterfly
  static_assert(f_radix(L, 0) == 32 && f_radix(L, 1) == 32 && RL >= 2, "radices 32, 32, L/1024");
  static_assert(T >= 64 && T <= 1024 && T % TG::S2 == 0, "whole waves, one sub-rotator entry per pass-0 column");
};

// LDS of one unit, in bytes: a component plane of L points (and, before the
// first exchange, the delay split, then the operands of M), the rotator
// tables, the 2-bit level pairs and the packed samples.  At 8192 real points
// 39.6 KB: four workgroups per CU.
template <int L, bool CPLX>
struct BLds {
  static constexpr int TAB = 4 * L;
  static constexpr int INC = TAB + TabGeom<L, CPLX>::NTAB * 8;
  static constexpr int LUT = INC + (rho_in_passes<L>() ? kNumIncs * 8 : 0);
  static constexpr int STAGE = LUT + (CPLX ? 0 : 128);
  static constexpr int BYTES = STAGE + (CPLX ? 0 : L / 2);
  static_assert(MatLds<CPLX>::BYTES <= 4 * L, "M's operands fit the plane");
};

// One component of the points between pass 1 and the last pass.
template <int L, bool CPLX, int COMP>
__device__ __forceinline__ void put_plane(const float2 (&v)[32], float *s, int j) {
  float *d = s + (j >> 5) * 1024 + (j & 31);
#pragma unroll
  for (int k = 0; k < 32; k++) d[32 * k] = COMP ? v[k].y : v[k].x;
}
// Butterfly CON j + bf of group g sits at v[(g CON + bf) RL ..]: its inputs are
// words CON (j + g T) + bf + k L/RL, CON neighbours in one LDS read.
template <int L, bool CPLX, int CON_, int COMP>
__device__ __forceinline__ void get_plane(float2 (&v)[32], const float *s, int j) {
  using G = BG<L, CPLX, CON_>;
  constexpr int CON = G::CON, RL = G::RL;
  typedef float row __attribute__((ext_vector_type(CON)));
#pragma unroll
  for (int g = 0; g < G::GRP; g++)
#pragma unroll
    for (int k = 0; k < RL; k++) {
      const row x = *reinterpret_cast<const row *>(s + CON * (j + g * G::T) + k * (L / RL));
#pragma unroll
      for (int bf = 0; bf < CON; bf++) {
        float2 &d = v[(g * CON + bf) * RL + k];
        if (COMP)
          d.y = x[bf];
        else
          d.x = x[bf];
      }
    }
}

// Last pass, butterflies I ..: twiddles, DFT, fractional-sample rotation of the
// kept outputs, which replace the butterfly's first ones.  w holds the powers
// of W_L^(CON j); butterfly CON j + bf + CON T g takes them times a constant.
template <int L, bool CPLX, int CON_, int I = 0>
__device__ __forceinline__ void last_butterflies(float2 (&v)[32], const Powers &w) {
  using G = BG<L, CPLX, CON_>;
  constexpr int CON = G::CON, RL = G::RL;
  if constexpr (I < G::NB) {
    constexpr int M = I % CON + CON * G::T * (I / CON);
    float2 *x = &v[I * RL];
    if constexpr (RL == 2) {
      x[1] = cmul(x[1], twc<L, M % L>(w.p1));
    } else {
      Powers u;
      u.p1 = twc<L, M % L>(w.p1);
      u.p2 = twc<L, 2 * M % L>(w.p2);
      u.p3 = twc<L, 3 * M % L>(w.p3);
      u.q0 = twc<L, 4 * M % L>(w.q0);
      u.q1 = twc<L, 8 * M % L>(w.q1);
      u.q2 = twc<L, 16 * M % L>(w.q2);
      times_powers<RL, 0>(x, u);
    }
    dft<RL>(x);
    last_butterflies<L, CPLX, CON_, I + 1>(v, w);
  }
}

// Unit u = station + nant * FFT (BOTH) or 2 * that + pol, on a workgroup of
// exactly BG::T threads (every thread calls it with the same u: it contains
// __syncthreads).  smem holds BLds::BYTES bytes, 16-byte aligned.
template <int L, bool CPLX, int OUT, bool BOTH>
__device__ __forceinline__ void fstage_big_item(const FParams &p, int u, unsigned char *smem) {
  // Neighbouring bins of a thread: 16 bytes, so that a wave's store covers whole
  // lines (four FP32 bins as two stores of 16 bytes, 32 apart per lane, took
  // 6.8 ms instead of 6.1 at 8192 points; 16-bit bins gain 5 % from two to four).
  constexpr int CON_ = out_bytes(OUT) == 8 ? 2 : 4;
  using G = BG<L, CPLX, CON_>;
  using TG = typename G::TG;
  using LD = BLds<L, CPLX>;
  constexpr int T = G::T, S = TG::S, S2 = TG::S2, NSTEPS = TG::NSTEPS, NCHAN = TG::NCHAN, TR = T / 32;
  constexpr int CON = G::CON, RL = G::RL;
  static_assert(!BOTH || !CPLX, "both polarisations in turn: 2-bit samples");
  float *splane = reinterpret_cast<float *>(smem);
  float2 *stab = reinterpret_cast<float2 *>(smem + LD::TAB);
  float2 *sinc = reinterpret_cast<float2 *>(smem + LD::INC);
  uint2 *slut = reinterpret_cast<uint2 *>(smem + LD::LUT);
  uint32_t *stage = reinterpret_cast<uint32_t *>(smem + LD::STAGE);

  const int tid = threadIdx.x;
  const int pol0 = BOTH ? 0 : u & 1;
  const int item = BOTH ? u : u >> 1;
  const int tl = item / p.nant;
  const int st = item % p.nant;
  const int t = p.t0 + tl * p.tstride;
  constexpr unsigned EB = out_bytes(OUT);
  unsigned char *out = out_base<OUT>(p) + ((size_t)item * 2 + pol0) * (NCHAN * EB);

  // The delay split (two FP64 divisions) on one wave; the others wait for it
  // at the barrier and leave the VALU to the other workgroups of the CU.
  struct Split {
    double frac, a, b;
    int offset, valid;
  };
  Split *ssplit = reinterpret_cast<Split *>(smem);
  if (T <= 64 || tid < 64) {
    Split w{0.0, 0.0, 0.0, 0, 0};
    w.valid = split_offset<L>(p, st, t, w.offset, w.frac, w.a, w.b) ? 1 : 0;
    if (tid == 0) {
      *ssplit = w;
      if (pol0 == 0 && OUT != OUT_POWER) p.valid[(size_t)st * p.numffts + t] = w.valid;
    }
  }
  __syncthreads();
  // The same for every thread of the workgroup: the branches below that
  // depend on it are uniform, so every __syncthreads is reached by all.
  const int offset = __builtin_amdgcn_readfirstlane(ssplit->offset);
  const bool valid = __builtin_amdgcn_readfirstlane(ssplit->valid) != 0;
  const double frac = ssplit->frac, a = ssplit->a, b = ssplit->b;
  if (!valid) {
    for (unsigned q = tid; q < (BOTH ? 2 : 1) * NCHAN; q += T) store_val<OUT>(out + q * EB, make_float2(0.f, 0.f), 1.f);
    return;
  }
  Pass0In<L, CPLX, true, 4> in;
  in.template load<T>((gbyte *)p.station[st], offset, tid, tid);
  fill_tables<L, CPLX>(p, frac, a, b, stab, tid, T, pass0_unscale<CPLX>());
  // by the second wave: the first has the tables' last entries
  if (rho_in_passes<L>() && (unsigned)(tid - 64) < kNumIncs) sinc[tid - 64] = inc_entry(p, a, 1.0 / L, tid - 64);
  if (!CPLX && tid < 16) slut[tid] = level_pair(tid);
  in.template put<T>(stage, tid);
  __syncthreads();
  build_matrix<CPLX, T>(smem, stab + S2, T / S2, p.twiddle, tid);
  __syncthreads();
  // M's operands for both polarisations (2-bit input: 16 registers)
  uint4 am[2][2];
  if constexpr (BOTH) {
#pragma unroll
    for (int i = 0; i < 4; i++) am[i >> 1][i & 1] = reinterpret_cast<const uint4 *>(smem)[64 * i + (tid & 63)];
  }

  auto one_pol = [&](const int pol) {
    // An opaque copy of the thread index (and an opaque zero offset) in
    // each polarisation's copy of this code keeps the compiler from sharing
    // the per-thread LDS and global addresses, the rotator, twiddle and
    // table reads and their products between the two copies, where they
    // would hold ~100 registers over the first FFT.
    int z = 0, j = threadIdx.x;
    if constexpr (BOTH) asm volatile("" : "+s"(z), "+v"(j));
    const float2 *sub = stab + z;
    const float2 *step = sub + S2;
    const float2 *fsub = step + NSTEPS;
    const float2 *fstep = fsub + S;
    const float2 *__restrict__ tw = p.twiddle + z;

    // ---- pass 0: columns j0 + tile of lane (c, g) ----
    const int c = j & 15, g = (j >> 4) & 3, j0 = (j & ~63) + 4 * c;
    floatx4 acc[4][2][2];
    in.fetch(stage + z, j);
    if constexpr (BOTH)
      in.matmul(acc, am, slut + z, pol);
    else
      in.matmul(acc, smem, slut + z, pol);
    finish_columns<L, CPLX, 4>(acc, sub, step, tw, j0, g);
    __syncthreads();  // M's operands (the last polarisation's points) are read
    // Exchange to pass 1, one component at a time: point 32 jj + r, in rows
    // of 8 chunks of 4 points at chunk position (r / 4) ^ (jj / 4 mod 8).
    // Eight neighbouring lanes of a 16-byte store then cover the 32 banks
    // once, and so do 32 lanes of a pass-1 load.
    float2 v[32];
    {
      const int r = j & 31, jr = j >> 5;
      const int b0 = 32 * jr + 4 * ((r >> 2) ^ ((jr >> 2) & 7)) + (r & 3);
#pragma unroll
      for (int comp = 0; comp < 2; comp++) {
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
          for (int rh = 0; rh < 2; rh++)
            *reinterpret_cast<floatx4 *>(splane + 32 * (j0 + e) + 4 * ((g ^ (c & 7)) ^ (4 * rh))) = acc[e][rh][comp];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 32; k++) {
          const float x = splane[(b0 ^ (4 * (((k * TR) >> 2) & 7))) + k * T];
          if (comp)
            v[k].y = x;
          else
            v[k].x = x;
        }
        __syncthreads();
      }
    }
    // ---- pass 1 and the last pass ----
    dft<32>(v);
    put_plane<L, CPLX, 0>(v, splane, j);
    __syncthreads();
    get_plane<L, CPLX, CON_, 0>(v, splane, j);
    __syncthreads();
    put_plane<L, CPLX, 1>(v, splane, j);
    __syncthreads();
    get_plane<L, CPLX, CON_, 1>(v, splane, j);
    constexpr int TWS = f_tw_step(L, 2);
    static_assert(CON % TWS == 0 || CON == 1, "the first butterfly's powers are in the table");
    last_butterflies<L, CPLX, CON_>(
        v, turn_powers<L>(load_powers<RL, f_tw_entries(L, 2), f_tw_off(L, 2)>(tw, (unsigned)j * (CON / TWS)), sinc + z));

    // outputs: bins q = CON (j + g T) + bf + k L/RL, q < nchan, CON neighbours
    // of a thread in one store
#pragma unroll
    for (int gr = 0; gr < G::GRP; gr++)
#pragma unroll
      for (int k = 0; k < G::KEEP; k++) {
        // q / S = CON j / S + a compile-time step: S divides CON T and L/RL,
        // CON divides S
        static_assert((CON * T) % S == 0 && (L / RL) % S == 0 && S % CON == 0, "table offsets");
        const int step0 = (CON * T * gr + k * (L / RL)) / S;
        const float2 fs = fstep[CON * j / S + step0];
        const unsigned q = (unsigned)(CON * j) + CON * T * gr + k * (L / RL);
        float2 y[CON];
        float sc[CON];
#pragma unroll
        for (int bf = 0; bf < CON; bf++) {
          const float2 fr = cmul(fsub[(CON * j) % S + bf], fs);  // fracsamprotator, fxkernel.cpp:614-625
          y[bf] = cmul(fr, v[(gr * CON + bf) * RL + k]);
          sc[bf] = bin_scale<OUT, NCHAN>(p, 2 * st + pol, q + bf);
        }
        store_row<OUT, CON>(out + ((unsigned)(BOTH ? pol : 0) * (NCHAN * EB) + q * EB), y, sc);
      }
  };
  one_pol(pol0);
  if constexpr (BOTH) one_pol(1);
}

}  // namespace fs
}  // namespace gxc
