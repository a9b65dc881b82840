// Transforms of G sequences of 2^LOG2L points with the values in registers: a thread holds
// 2^LOGR points (16 unless said), runs whole butterflies of that radix (fft_lds.hpp) and
// hands them to the next stage through LDS, so that a 256-point sequence crosses LDS once
// where the radix-4 stages cross it four times; the first stage's inputs and the last
// stage's outputs stay in registers for the caller to load, use and store. The stage of a
// smaller radix for what remains of L runs last, or first: the values a transform ends
// with are then the very ones the opposite transform starts from. A workgroup of more
// threads than the butterflies need (THREADS) leaves the others idle in the stages.
//
// The LDS layout follows the way the caller's lanes run. Column: neighbouring lanes hold
// neighbouring sequences (a strided axis); points are stored sequence-fastest, so that
// every access moves whole runs of G points. Row: neighbouring lanes hold neighbouring
// points of one sequence (a contiguous axis); rows are padded by one point in 16, as a
// radix-16 stage stores its outputs 16 points apart.
#pragma once

#include "fft_lds.hpp"

namespace sp {

template <int LOG2L, int G, bool Column, bool RestFirst, int LOGR = 4, int THREADS = 0>
struct RegsFft {
  static constexpr int L = 1 << LOG2L;
  static constexpr int E = L * G;
  static constexpr int MAX = 1 << LOGR;
  static constexpr int NT = THREADS > 0 ? THREADS : (E >= MAX ? E / MAX : 1);
  static constexpr int full = LOG2L / LOGR;
  static constexpr int rest = (1 << LOG2L) >> (LOGR * full);
  static constexpr int stages = full + (rest > 1 ? 1 : 0);
  static constexpr int STRIDE = padded(L);
  static constexpr int LDS_POINTS = Column ? E : G * STRIDE;
  static_assert(NT <= 1024, "a workgroup has at most 1024 threads");

  static constexpr int radix(int stage) {
    return rest == 1 ? MAX
                     : (RestFirst ? (stage == 0 ? rest : MAX) : (stage < full ? MAX : rest));
  }

  // The butterflies a thread runs in a stage of radix R: `b` counts them over the
  // workgroup, each with inputs i + j L/R of sequence s.
  template <int R>
  static constexpr int per() {
    return (E / R + NT - 1) / NT;
  }
  template <int R>
  using Regs = cplx[per<R>()][R];
  using First = Regs<radix(0)>;
  using Last = Regs<radix(stages - 1)>;

  template <int R>
  static __device__ __forceinline__ int sequence(int b) {
    return Column ? b % G : b / (L / R);
  }
  template <int R>
  static __device__ __forceinline__ int input(int b) {
    return Column ? b / G : b % (L / R);
  }
  static __device__ __forceinline__ int slot(int s, int point) {
    return Column ? point * G + s : s * STRIDE + padded(point);
  }

  // Calls f(value, sequence, point) for each input of the first stage.
  template <class F>
  static __device__ __forceinline__ void inputs(First& v, F f) {
    constexpr int R = radix(0);
#pragma unroll
    for (int r = 0; r < per<R>(); ++r) {
      const int b = static_cast<int>(threadIdx.x) + r * NT;
      if (E / R % NT == 0 || b < E / R) {
        const int s = sequence<R>(b), i = input<R>(b);
#pragma unroll
        for (int j = 0; j < R; ++j) f(v[r][j], s, i + j * (L / R));
      }
    }
  }

  // Calls f(value, sequence, point) for each output of the last stage.
  template <class F>
  static __device__ __forceinline__ void outputs(Last& v, F f) {
    constexpr int R = radix(stages - 1);
#pragma unroll
    for (int r = 0; r < per<R>(); ++r) {
      const int b = static_cast<int>(threadIdx.x) + r * NT;
      if (E / R % NT == 0 || b < E / R) {
        const int s = sequence<R>(b), i = input<R>(b);
#pragma unroll
        for (int j = 0; j < R; ++j) f(v[r][out_at<R>(j)], s, i + j * (L / R));
      }
    }
  }

  // The stages' twiddles, loaded ahead of the data they turn (a stage would otherwise wait
  // for its own after each barrier): worth their registers in launches whose time is
  // latency.
  struct Twiddles {
    cplx w[stages > 1 ? stages - 1 : 1][MAX];
  };
  static __device__ __forceinline__ void twiddles(Twiddles& t, const cplx* __restrict__ tw,
                                                  int sign) {
    twiddles_from<1>(t, tw, sign);
  }
  static __device__ __forceinline__ void run(First& in, Last& out, cplx* lds, const Twiddles& t,
                                             int sign) {
    stage<0>(in, out, lds, &t, nullptr, sign);
  }

  // The transform: `in` is consumed, `out` receives the last stage's values, `lds` holds
  // LDS_POINTS points that nothing else reads or writes until the workgroup's next
  // barrier. `sign` is a constant at every call, so its selections fold.
  static __device__ __forceinline__ void run(First& in, Last& out, cplx* lds,
                                             const cplx* __restrict__ tw, int sign) {
    stage<0>(in, out, lds, static_cast<const Twiddles*>(nullptr), tw, sign);
  }

 private:
  static constexpr int span(int stage) {
    int p = 1;
    for (int k = 0; k < stage; ++k) p *= radix(k);
    return p;
  }

  template <int S>
  static __device__ __forceinline__ void twiddles_from(Twiddles& t, const cplx* __restrict__ tw,
                                                       int sign) {
    if constexpr (S < stages) {
      constexpr int R = radix(S), p = span(S), step = L / (p * R);
#pragma unroll
      for (int r = 0; r < per<R>(); ++r) {
        const int b = static_cast<int>(threadIdx.x) + r * NT;
        if (E / R % NT == 0 || b < E / R) {
          const int k = input<R>(b) & (p - 1);
#pragma unroll
          for (int j = 1; j < R; ++j)
            t.w[S - 1][r * (R - 1) + j - 1] = twiddle(tw, j * k * step, sign);
        }
      }
      twiddles_from<S + 1>(t, tw, sign);
    }
  }

  template <int S>
  static __device__ __forceinline__ void stage(Regs<radix(S)>& v, Last& out, cplx* lds,
                                               const Twiddles* held, const cplx* __restrict__ tw,
                                               int sign) {
    constexpr int R = radix(S), p = span(S), step = L / (p * R);
#pragma unroll
    for (int r = 0; r < per<R>(); ++r) {
      const int b = static_cast<int>(threadIdx.x) + r * NT;
      if (E / R % NT == 0 || b < E / R) {
        const int k = input<R>(b) & (p - 1);
        if constexpr (p > 1)
#pragma unroll
          for (int j = 1; j < R; ++j)
            v[r][j] = mul(v[r][j], held ? held->w[S - 1][r * (R - 1) + j - 1]
                                        : twiddle(tw, j * k * step, sign));
        dft<R>(v[r], sign);
      }
    }
    if constexpr (S == stages - 1) {
#pragma unroll
      for (int r = 0; r < per<R>(); ++r)
#pragma unroll
        for (int j = 0; j < R; ++j) out[r][j] = v[r][j];
    } else {
      constexpr int RN = radix(S + 1);
      if constexpr (S > 0) __syncthreads();  // the last hand-over's reads are done
#pragma unroll
      for (int r = 0; r < per<R>(); ++r) {
        const int b = static_cast<int>(threadIdx.x) + r * NT;
        if (E / R % NT == 0 || b < E / R) {
          const int s = sequence<R>(b), i = input<R>(b), k = i & (p - 1);
#pragma unroll
          for (int j = 0; j < R; ++j) lds[slot(s, (i - k) * R + k + j * p)] = v[r][out_at<R>(j)];
        }
      }
      __syncthreads();
      Regs<RN> next;
#pragma unroll
      for (int r = 0; r < per<RN>(); ++r) {
        const int b = static_cast<int>(threadIdx.x) + r * NT;
        if (E / RN % NT == 0 || b < E / RN) {
          const int s = sequence<RN>(b), i = input<RN>(b);
#pragma unroll
          for (int j = 0; j < RN; ++j) next[r][j] = lds[slot(s, i + j * (L / RN))];
        }
      }
      stage<S + 1>(next, out, lds, held, tw, sign);
    }
  }
};

}  // namespace sp
