// The F-stage for FFT lengths 64..1024 as a device function over one
// workgroup's items (station, FFT).
//
// Per item, fused so the packed samples are read once and the spectra
// written once:
//   1. FP64 delay model and integer/fractional split (fxkernel.cpp:288-309,
//      425-440), one item per lane of the first wave.
//   2. Fringe-rotator and fractional-sample tables (fxkernel.cpp:498-567,
//      595-634) in LDS, built by the item's threads for both polarisations.
//   3. First FFT pass, radix 16, from the packed samples (fstage_pass0.hpp).
//   4. Remaining Stockham passes of radix 4..16 through LDS.
//   5. Last pass writes only bins < nchan, multiplied by the fractional
//      sample rotator, as coalesced stores to spectra[t][2*station+pol][chan].
//
// What bounds it is issue and latency together: with two waves ready, a SIMD
// issues an FP32 or simple integer instruction on VGPRs every ~2.4 cycles,
// one wave alone every ~5, so waves in flight count.  A thread therefore
// holds 16 points of one polarisation (32 registers), the two polarisations
// of an item sit on neighbouring threads, and points are exchanged one
// component plane at a time: 64 registers and 4.5 bytes of LDS per point, 8
// waves per SIMD.  Against one thread per 16 points of both polarisations (3-4
// waves): 32 stations x 1024 complex channels 1.15 -> 0.79 ms, 5 stations x 512
// channels 0.42 -> 0.27 ms (before fstage_1k.hpp took real input of 1024 points).
#pragma once

#include "fstage_pass0.hpp"

namespace gxc {
namespace fs {

// Compile-time geometry for FFT length L.
template <int L, bool CPLX>
struct QG {
  using TG = TabGeom<L, CPLX>;
  static constexpr int NCHAN = TG::NCHAN, S = TG::S, S2 = TG::S2, NSTEPS = TG::NSTEPS, NTAB = TG::NTAB;
  static constexpr int T = L / 16;          // threads per polarisation of an item
  static constexpr int radix(int p) { return f_radix(L, p); }
  static constexpr int ns(int p) { return f_ns(L, p); }
  static constexpr int NPASS = f_npass(L);
  // LDS word of point i of a component plane: 4 words of padding per 32, so
  // that 16-byte stores of pass 0 by 8 neighbouring lanes, the stores of the
  // middle pass and all loads fall in 32 distinct banks per 32 lanes, and the
  // points of one thread sit at compile-time offsets (strides are multiples of
  // the padding period, or the thread's first point lies in the first 16
  // words).
  __device__ static constexpr int pad(int i) { return i + ((i >> 5) << 2); }
  // planes of neighbouring polarisations: T words apart modulo the 32 banks
  // where a half wave holds several of them
  static constexpr int PLANE = pad(L) + (T >= 32 ? 0 : (T + 32 - pad(L) % 32) % 32);
  static_assert(ns(NPASS) == L && PLANE % 4 == 0, "radix schedule");
  static_assert(L >= 64 && L <= 1024, "FFT lengths 64..1024");
};

// Delay split of one item (split_offset's results).
struct Split {
  double frac, a, b;
  int offset, valid;
};

// LDS of one workgroup of IPW items, in bytes.
template <int L, bool CPLX, int IPW>
struct QLds {
  using G = QG<L, CPLX>;
  static constexpr int PLANES = 4 * IPW * 2 * G::PLANE;
  static constexpr int TAB = PLANES;
  static constexpr int LUT = TAB + IPW * G::NTAB * 8;
  static constexpr int BYTES = LUT + (CPLX ? 0 : 16);
  // the delay splits lie where the first exchange comes later
  static_assert(IPW * (int)sizeof(Split) <= PLANES, "the delay splits fit");
};

// Stores of one component of pass P's outputs (P >= 1) and loads of its inputs.
template <int L, bool CPLX, int P, int COMP>
__device__ __forceinline__ void put16(const float2 (&v)[16], float *s, int j) {
  using G = QG<L, CPLX>;
  constexpr int R = G::radix(P), NS = G::ns(P), NB = 16 / R, T = G::T;
#pragma unroll
  for (int bf = 0; bf < NB; bf++) {
    const int b = j + bf * T;
    float *d = s + G::pad((b / NS) * (NS * R) + (b % NS));
#pragma unroll
    for (int k = 0; k < R; k++) d[G::pad(k * NS)] = COMP ? v[bf * R + k].y : v[bf * R + k].x;
  }
}

template <int L, bool CPLX, int P, int COMP>
__device__ __forceinline__ void get16(float2 (&v)[16], const float *s, int j) {
  using G = QG<L, CPLX>;
  constexpr int R = G::radix(P), NB = 16 / R, T = G::T, STR = L / R;
#pragma unroll
  for (int bf = 0; bf < NB; bf++) {
    const float *d = s + G::pad(j + bf * T);
#pragma unroll
    for (int k = 0; k < R; k++) {
      const float x = d[G::pad(k * STR)];
      if (COMP)
        v[bf * R + k].y = x;
      else
        v[bf * R + k].x = x;
    }
  }
}

// Twiddles and butterfly BF of pass P.
// Butterfly BF's index is j + BF*T: the same modulo NS where NS divides T,
// else (last pass) its twiddles are butterfly 0's times W_L^(BF T power), a
// constant W_16^(BF power).
template <int L, bool CPLX, int P, int BF>
__device__ __forceinline__ void butterfly16(float2 *v, const Powers &w) {
  using G = QG<L, CPLX>;
  constexpr int R = G::radix(P), NS = G::ns(P), T = G::T;
  if constexpr (BF == 0 || T % NS == 0) {
    times_powers<R, 0>(v, w);
  } else {
    static_assert(NS * R == L, "last pass");
    Powers u;
    u.p1 = twc<16, BF>(w.p1);
    u.p2 = twc<16, 2 * BF>(w.p2);
    u.p3 = twc<16, 3 * BF>(w.p3);
    u.q0 = u.q1 = u.q2 = twc<16, 4 * BF>(w.q0);
    static_assert(R <= 8, "powers up to 4");
    times_powers<R, 0>(v, u);
  }
  dft<R>(v);
}
template <int L, bool CPLX, int P>
__device__ __forceinline__ Powers powers16(int j, const float2 *__restrict__ tw) {
  using G = QG<L, CPLX>;
  constexpr int R = G::radix(P), NS = G::ns(P);
  return load_powers<R, NS, f_tw_off(L, P)>(tw, (unsigned)j % NS);
}
template <int L, bool CPLX, int P, int BF = 0>
__device__ __forceinline__ void pass16(float2 (&v)[16], const Powers &w) {
  constexpr int R = QG<L, CPLX>::radix(P);
  if constexpr (BF < 16 / R) {
    butterfly16<L, CPLX, P, BF>(&v[BF * R], w);
    pass16<L, CPLX, P, BF + 1>(v, w);
  }
}

// Last pass, butterflies BF ..: outputs are bins q = b + k*(L/R), of which
// q < nchan are kept, times the fractional-sample rotator
// (fxkernel.cpp:614-625).  One butterfly after the other: the scheduler
// would otherwise hold both butterflies' twiddles and factors at once.
template <int L, bool CPLX, int OUT, int BF = 0>
__device__ __forceinline__ void last16(const FParams &p, float2 (&v)[16], const Powers &w, int j, const float2 *fsub,
                                       const float2 *fstep, unsigned char *out0, unsigned rowoff, int srow, bool store,
                                       bool valid) {
  using G = QG<L, CPLX>;
  constexpr int P = G::NPASS - 1, R = G::radix(P), KEEP = CPLX ? R : R / 2, T = G::T, S = G::S;
  constexpr unsigned EB = out_bytes(OUT);
  if constexpr (BF < 16 / R) {
    if constexpr (BF > 0) __builtin_amdgcn_sched_barrier(0);
    butterfly16<L, CPLX, P, BF>(&v[BF * R], w);
    if (store) {
#pragma unroll
      for (int k = 0; k < KEEP; k++) {
        const int q = j + BF * T + k * (L / R);
        // q % S = j % S and q / S = j / S + a compile-time step when S
        // divides T and L/R
        const float2 fr = (T % S == 0 && (L / R) % S == 0) ? cmul(fsub[j % S], fstep[j / S + (BF * T + k * (L / R)) / S])
                                                           : cmul(fsub[q % S], fstep[q / S]);
        float2 y = cmul(fr, v[BF * R + k]);
        if (!valid) y = make_float2(0.f, 0.f);
        store_val<OUT, (T * EB >= 64)>(out0 + (rowoff + (unsigned)q * EB), y, bin_scale<OUT, G::NCHAN>(p, srow, q));
      }
    }
    last16<L, CPLX, OUT, BF + 1>(p, v, w, j, fsub, fstep, out0, rowoff, srow, store, valid);
  }
}

// Items blk*IPW .. of one launch (item = station + nant * FFT) with both
// polarisations on a workgroup of exactly IPW * 2 T threads (every thread
// calls it with the same blk: it contains __syncthreads).  smem holds
// QLds::BYTES bytes, 16-byte aligned.
template <int L, bool CPLX, int OUT, int IPW>
__device__ __forceinline__ void fstage16_item(const FParams &p, int blk, unsigned char *smem) {
  using G = QG<L, CPLX>;
  using LD = QLds<L, CPLX, IPW>;
  constexpr int T = G::T, S = G::S, S2 = G::S2, NSTEPS = G::NSTEPS, NCHAN = G::NCHAN;
  constexpr bool WAVE = T >= 64;  // a wave holds one polarisation of one item
  const int tid = threadIdx.x;
  const int j = tid & (T - 1);
  int grp = tid / T;  // polarisation + 2 * item of the workgroup
  if (WAVE) grp = __builtin_amdgcn_readfirstlane(grp);
  const int li = grp >> 1, pol = grp & 1;
  const int item0 = blk * IPW;
  const int nitems = p.nant * p.nt;

  Split *ssplit = reinterpret_cast<Split *>(smem);
  if (tid < IPW) {
    Split w{0.0, 0.0, 0.0, 0, 0};
    const int item = item0 + tid;
    if (item < nitems) {
      const int tl = item / p.nant, st = item - tl * p.nant, t = p.t0 + tl * p.tstride;
      w.valid = split_offset<L>(p, st, t, w.offset, w.frac, w.a, w.b) ? 1 : 0;
      if (OUT != OUT_POWER) p.valid[(size_t)st * p.numffts + t] = w.valid;
    }
    ssplit[tid] = w;
  }
  __syncthreads();
  const int item = item0 + li;
  const int st = item % p.nant;
  int offset = ssplit[li].offset;
  int ok = ssplit[li].valid;
  if (WAVE) {
    offset = __builtin_amdgcn_readfirstlane(offset);
    ok = __builtin_amdgcn_readfirstlane(ok);
  }
  const bool valid = ok != 0;

  float2 *stab = reinterpret_cast<float2 *>(smem + LD::TAB) + li * G::NTAB;
  float *splane = reinterpret_cast<float *>(smem) + grp * G::PLANE;
  const float2 *sub = stab, *step = sub + S2, *fsub = step + NSTEPS, *fstep = fsub + S;

  // Packed samples, requested before the table build.
  Pass0In<L, CPLX, false, 0> in;
  if (valid) {
    in.load((gbyte *)p.station[st], offset, j);
    fill_tables<L, CPLX>(p, ssplit[li].frac, ssplit[li].a, ssplit[li].b, stab, tid - li * 2 * T, 2 * T);
  }
  float *slut = reinterpret_cast<float *>(smem + LD::LUT);
  if (!CPLX && tid < 4) slut[tid] = tid == 0 ? -kHiMag : tid == 1 ? -1.0f : tid == 2 ? 1.0f : kHiMag;
  __syncthreads();

  float2 v[16];
  if (valid) {
    in.rotate(v, sub, step, slut, pol, j);
  } else {
#pragma unroll
    for (int k = 0; k < 16; k++) v[k] = make_float2(0.f, 0.f);
  }
  dft<16>(v);
#pragma unroll
  for (int comp = 0; comp < 2; comp++) {
    float *d = splane + G::pad(16 * j);
#pragma unroll
    for (int ch = 0; ch < 4; ch++)
      *reinterpret_cast<floatx4 *>(d + 4 * ch) =
          comp ? floatx4{v[4 * ch].y, v[4 * ch + 1].y, v[4 * ch + 2].y, v[4 * ch + 3].y}
               : floatx4{v[4 * ch].x, v[4 * ch + 1].x, v[4 * ch + 2].x, v[4 * ch + 3].x};
    __syncthreads();
    if (comp)
      get16<L, CPLX, 1, 1>(v, splane, j);
    else
      get16<L, CPLX, 1, 0>(v, splane, j);
    __syncthreads();
  }
  if constexpr (G::NPASS > 2) {
    pass16<L, CPLX, 1>(v, powers16<L, CPLX, 1>(j, p.twiddle));
    put16<L, CPLX, 1, 0>(v, splane, j);
    __syncthreads();
    get16<L, CPLX, 2, 0>(v, splane, j);
    __syncthreads();
    put16<L, CPLX, 1, 1>(v, splane, j);
    __syncthreads();
    get16<L, CPLX, 2, 1>(v, splane, j);
  }
  constexpr unsigned EB = out_bytes(OUT);
  last16<L, CPLX, OUT>(p, v, powers16<L, CPLX, G::NPASS - 1>(j, p.twiddle), j, fsub, fstep,
                       out_base<OUT>(p) + (size_t)(2 * item0) * (NCHAN * EB), (unsigned)grp * (NCHAN * EB),
                       2 * st + pol, item < nitems, valid);
}

}  // namespace fs
}  // namespace gxc
