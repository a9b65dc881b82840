// The envelope route's stages as transforms joined at their ends, FP64, for gfx950.
//
// A stage is four transforms of T points (two without a Raman response) with pointwise
// work between them: entry -> inverse -> Raman drive -> forward -> kernel product ->
// inverse -> response -> forward -> finish. At the sizes of a fibre's grid each launch
// costs more than its work, so the launches are what to save. A transform of T = L S
// points is split in two passes (columns of L points at stride S, the W_T twiddle, then
// rows), and its second pass leaves workgroup s with the points k S + s (k < L): exactly a
// column of the next transform, where that one is split the other way round. The second
// pass of one transform, the pointwise work and the first pass of the next are therefore
// one kernel over L-point sequences that never leaves registers and LDS, and a stage is
// four launches (two without Raman) instead of twelve (six). Every kernel has one form:
//
//   read row s of the input (L contiguous points), transform, work at the points
//   k S + s, transform, times W_T^(s k), write point k to row k (contiguous in s).
//
// The Raman convolution over the doubled grid keeps T points without pairing bins: with
// w = W_4T^t the drive d (zero from T on) and the response h = (h1, h2) of 2T samples give
//   Re[ conj(w_t) IFFT_T( FFT_T(w d) FFT_T(w (h1 + i h2)) )_t ]
//     = sum_{s <= t} d_s h1_{t-s} + sum_{s > t} d_s h2_{T+t-s},
// the circular convolution of 2T points on its first T: wrapping round T turns by
// w_T = -i, and the i before h2 turns its wrapped part back.
//
// What bounds a kernel is latency (its launch, one read of the input, the stages' LDS
// hand-overs): 4 to 7 us each on 2^14 samples. An attempt of six stages with Raman on 2^13
// bins and 2^14 samples took 322 us in 76 launches and takes 137 in 26; a trial of seven on
// 2^16 bins and 2^17 samples took 845 and takes 427.
#include "kernels.hpp"

#include "fft_regs.hpp"

namespace sp {

namespace {

__device__ inline cplx phase_sum(const double* w, const cplx* terms, int n_terms, long stride,
                                 long at) {
  cplx total = make(0.0, 0.0);
  for (int t = 0; t < n_terms; ++t) total = add(total, scale(w[t], terms[t * stride + at]));
  return total;
}

enum Kind { kEntry, kDrive, kProduct, kResponse, kFinish, kAccept };

// ------------------------------------------------------------------ one coarse bin

// What a bin's stage input needs beside its last derivative, formed while the transform
// runs: u = fwd (y + dz (sum_j<n a_j k_j)) + noise.
struct BinEntry {
  cplx fwd, back, y, comb, noise;
};

__device__ inline BinEntry bin_entry(const EnvStage& a, int stage, int known, int b) {
  const DeviceProblem& P = a.P;
  const StageRow& row = a.R->stage[stage];
  BinEntry e;
  e.y = a.y[b];
  if (a.commit) {
    e.y = P.active[b] ? a.adv[b] : make(0.0, 0.0);
    a.y[b] = e.y;
  }
  if (a.recycle) a.k[b] = a.recycled[b];
  e.comb = make(0.0, 0.0);
  for (int j = 0; j < known; ++j)
    e.comb = add(e.comb, scale(P.tab_a[stage * P.n_stages + j],
                               a.k[static_cast<long>(j) * P.N + b]));
  const cplx dphi = phase_sum(row.phi_w, P.phi, P.n_phi, P.N, b);
  cexp_pair(dphi, &e.fwd, &e.back);
  e.noise = make(0.0, 0.0);
  if (P.noise_modified) {
    double phase = 0.0;
    for (int t = 0; t < P.n_phi; ++t)
      phase = phase + row.noise_w[t] * P.phi[static_cast<long>(t) * P.N + b].y;
    double s, co;
    sincos(phase, &s, &co);
    e.noise = mul(P.noise[b], make(co, s));
  }
  return e;
}

// The stage's input at the bin (1/T folded in for the inverse transform); the factor its
// derivative will be turned back by is kept.
__device__ inline cplx bin_input(const EnvStage& a, const BinEntry& e, int b) {
  a.einv[b] = e.back;
  cplx u = mul(e.fwd, add(e.y, scale(a.R->dz, e.comb)));
  if (a.P.noise_modified) u = add(u, e.noise);
  return scale(a.P.inv_T, u);
}

// Stage `stage`'s derivative at a bin from its transformed response: k = einv (p W P~ + A),
// the absorber's term unscaled on the active band
// (src/solprop/backends/numpy_ref/passes/stepping.py:88-145).
struct BinFinish {
  cplx pref, einv;
  bool absorbed;
};

__device__ inline BinFinish bin_finish(const EnvStage& a, int stage, int b) {
  const DeviceProblem& P = a.P;
  BinFinish f;
  f.pref = scale(P.omega_window[b], phase_sum(a.R->stage[stage].pref_w, P.pref, P.n_pref, P.N, b));
  f.einv = a.einv[b];
  f.absorbed = P.absorber_stream >= 0 && P.active[b];
  return f;
}

__device__ inline cplx bin_derivative(const EnvStage& a, const BinFinish& f, int stage, int b,
                                      cplx response, cplx absorber) {
  cplx v = mul(f.pref, response);
  if (f.absorbed) v = add(v, absorber);
  v = mul(f.einv, v);
  a.k[static_cast<long>(stage) * a.P.N + b] = v;
  return v;
}

// ------------------------------------------------------------------ the kernels

// Sequences a workgroup owns (log2): 2^9 points (fewer on the shortest sequences, whose
// count is no more than L / 2), and 2^10 on sequences of 512 points, and of 256 in the
// kernels with work at the bins, which belong to grids of 2^16 samples or more: there the
// chip is full all the same, and neighbouring sequences share the lines that a stored or
// gathered point would touch alone. A march of 20 attempts on 2^15 samples takes 3.23 ms
// at 2^9 points, 3.61 at 2^8 and 3.39 at 2^10; a trial on 2^17, 506, 567 and 473 us.
// Sequences of 1024 points or more (2^19 samples on) take 2^12 points, what LDS holds: a
// lone sequence moved a line for every point it stored or gathered. A trial on 2^20 bins
// took 1.83 ms; in the order of sequence_group 0.91 at 2^10 points, 0.65 at 2^11 and 0.55
// at 2^12 (1.32 with the transforms and the work at the bins apart).
constexpr int env_log2g(int log2l, bool bins) {
  const int points = log2l >= 10 ? 12 : (log2l >= (bins ? 8 : 9) ? 10 : 9);
  const int want = points - log2l, most = log2l > 1 ? log2l - 1 : 0;
  const int g = want < 0 ? 0 : want;
  return g < most ? g : most;
}

// The group of sequences a workgroup takes. Workgroups go to the eight XCDs in turn; each
// XCD takes a consecutive run of groups, so that the workgroups that share a line share an
// L2 (in launch order every XCD fetched, and wrote in parts, every line of the strided
// side). For sequences of 256 points or more, whose launches hold a multiple of 32 groups:
// below, a launch is too short for it (2^14 samples 93 us either way). A trial on 2^16 bins
// and samples 133 -> 112 us, on 2^19 610 -> 366.
template <int LOG2L>
__device__ inline int sequence_group() {
  const int b = static_cast<int>(blockIdx.x), n = static_cast<int>(gridDim.x);
  return LOG2L >= 8 ? b % 8 * (n / 8) + b / 8 : b;
}

// The kernels with work at the bins (two exponentials and a sine and cosine each) take a
// thread a point (one to four on the long sequences), the others a thread eight points.
template <int LOG2L, int Kind>
struct EnvShape {
  static constexpr int L = 1 << LOG2L;
  static constexpr bool bins = Kind == kEntry || Kind == kFinish || Kind == kAccept;
  static constexpr int G = 1 << env_log2g(LOG2L, bins);
  static constexpr int E = L * G;
  // A long strided side moves whole lines, 64 bytes, unless LDS holds no more sequences.
  static_assert(LOG2L < 10 || G >= 4 || E == 4096);
  static constexpr int THREADS = bins ? (E < 1024 ? E : 1024) : (E >= 8 ? E / 8 : 1);
  static constexpr bool held = LOG2L <= 9 && THREADS <= 512;  // twiddles in registers
  using First = RegsFft<LOG2L, G, true, false, 3, THREADS>;
  using Second = RegsFft<LOG2L, G, true, true, 3, THREADS>;
};

template <int LOG2L, int Kind>
__global__ void __launch_bounds__((EnvShape<LOG2L, Kind>::THREADS))
    env_kernel(EnvStage a, int stage) {
  using H = EnvShape<LOG2L, Kind>;
  using I = typename H::First;
  using F = typename H::Second;
  constexpr int L = H::L, G = H::G, E = H::E, NT = H::THREADS;
  constexpr int first_sign = Kind == kDrive || Kind == kResponse ? +1 : -1;
  constexpr int second_sign = -first_sign;
  constexpr int POINTS = (E + NT - 1) / NT;  // points a thread takes at the bins
  const DeviceProblem& P = a.P;
  const int tid = threadIdx.x;
  const int group = sequence_group<LOG2L>();
  const int s0 = group * G;
  const int S = P.T >> LOG2L;
  const cplx* tw = a.roots_l[LOG2L == a.log2n1 ? 0 : 1];
  __shared__ cplx lds[E];

  // The rows as the input holds them.
  typename I::First v;
  typename I::Last w;
  typename F::First u;
  typename F::Last z;
  if constexpr (Kind != kEntry)
    I::inputs(v, [&](cplx& x, int s, int j) { x = a.in[static_cast<long>(s0 + s) * L + j]; });

  // What does not wait for them: the twiddles, and at the bins all but the response.
  [[maybe_unused]] typename I::Twiddles first_tw;
  [[maybe_unused]] typename F::Twiddles second_tw;
  [[maybe_unused]] typename F::Last turn;
  auto turn_at = [&](cplx& x, int s, int k) { x = twiddle(a.roots, (s0 + s) * k, second_sign); };
  if constexpr (H::held) {
    if constexpr (Kind != kEntry) I::twiddles(first_tw, tw, first_sign);
    if constexpr (Kind != kAccept) {
      F::twiddles(second_tw, tw, second_sign);
      F::outputs(turn, turn_at);
    }
  }
  auto fine_of = [&](int e) { return (e / G) * S + s0 + e % G; };
  [[maybe_unused]] BinEntry entry;
  [[maybe_unused]] BinFinish finish;
  [[maybe_unused]] int bin = -1;
  // A thread a point (POINTS == 1): its bin's operands are read ahead.
  auto ahead = [&](int e) {
    bin = P.fine_to_coarse[fine_of(e)];
    if (bin < 0) return;
    if constexpr (Kind == kFinish) finish = bin_finish(a, stage - 1, bin);
    if constexpr (Kind == kAccept) finish = bin_finish(a, stage, bin);
    if constexpr (Kind == kEntry) entry = bin_entry(a, stage, stage, bin);
    if constexpr (Kind == kFinish) entry = bin_entry(a, stage, stage - 1, bin);
  };
  if constexpr (H::bins && POINTS == 1) ahead(tid);

  auto transform_in = [&](int row) {
    if (row > 0)
      I::inputs(v, [&](cplx& x, int s, int j) {
        x = a.in[static_cast<long>(row) * P.T + static_cast<long>(s0 + s) * L + j];
      });
    if constexpr (H::held)
      I::run(v, w, lds, first_tw, first_sign);
    else
      I::run(v, w, lds, tw, first_sign);
  };
  auto transform_out = [&](int row) {
    if constexpr (H::held)
      F::run(u, z, lds, second_tw, second_sign);
    else
      F::run(u, z, lds, tw, second_sign);
    if constexpr (!H::held) F::outputs(turn, turn_at);
    constexpr int R = F::radix(F::stages - 1);
#pragma unroll
    for (int r = 0; r < F::template per<R>(); ++r)
#pragma unroll
      for (int j = 0; j < R; ++j) z[r][j] = mul(z[r][j], turn[r][j]);
    F::outputs(z, [&](cplx& x, int s, int k) {
      a.out[static_cast<long>(row) * P.T + static_cast<long>(k) * S + s0 + s] = x;
    });
  };
  // The first transform's outputs as the second's inputs, through f(value, sequence, point).
  auto through = [&](auto f) {
    I::outputs(w, f);
    constexpr int R = F::radix(0);
#pragma unroll
    for (int r = 0; r < F::template per<R>(); ++r)
#pragma unroll
      for (int j = 0; j < R; ++j) u[r][j] = w[r][out_at<R>(j)];
  };

  if constexpr (Kind == kDrive) {
    transform_in(0);
    const double amplitude = P.synthesis[0] * a.R->stage[stage].taper;
    through([&](cplx& x, int s, int k) {
      a.field[static_cast<long>(k) * S + s0 + s] = x;
      const double d = 0.5 * norm2(scale(amplitude, x));
      x = scale(d, a.twist[static_cast<long>(k) * S + s0 + s]);
    });
    __syncthreads();
    transform_out(0);
  } else if constexpr (Kind == kProduct) {
    transform_in(0);
    through([&](cplx& x, int s, int k) {
      x = mul(x, a.kernel[static_cast<long>(k) * S + s0 + s]);
    });
    __syncthreads();
    transform_out(0);
  } else if constexpr (Kind == kResponse) {
    transform_in(0);
    const StageRow& row = a.R->stage[stage];
    const double amplitude = P.synthesis[0] * row.taper, back = P.projection[0] / row.taper;
    const double kerr = P.has_kerr ? P.kerr_coefficient * row.density : 0.0;
    const double raman = P.raman_epsilon0 * row.density;
    typename I::Last held;
    I::outputs(held, [&](cplx& x, int s, int k) {
      if (P.n_raman > 0) x = a.field[static_cast<long>(k) * S + s0 + s];
    });
    constexpr int R = I::radix(I::stages - 1);
#pragma unroll
    for (int r = 0; r < I::template per<R>(); ++r)
#pragma unroll
      for (int j = 0; j < R; ++j) {
        const int at = out_at<R>(j);
        if (P.n_raman <= 0) held[r][at] = w[r][at];
        const int b = tid + r * NT;
        if (!(E / R % NT == 0 || b < E / R)) continue;
        const long t = static_cast<long>(I::template input<R>(b) + j * (L / R)) * S + s0 +
                       I::template sequence<R>(b);
        const cplx e = scale(amplitude, held[r][at]);
        cplx pol = make(0.0, 0.0);
        if (P.has_kerr) {
          const cplx squares = mul(e, e);
          const cplx self = scale(P.kerr_self * norm2(e), e);
          const cplx conjugate = mul(scale(P.kerr_conjugate, squares), conj(e));
          pol = add(pol, scale(kerr, add(self, conjugate)));
        }
        if (P.n_raman > 0) {
          const cplx g = a.twist[t], c = w[r][at];
          const double cv = (g.x * c.x + g.y * c.y) * P.inv_T;  // Re(conj(g) c) / T
          pol = add(pol, scale(cv, scale(raman, e)));
        }
        u[r][j] = scale(back, scale(P.t_window[t], pol));
      }
    __syncthreads();
    transform_out(0);
    if (P.absorber_stream >= 0) {
      // The in-stage absorber's term from the modal field, transformed as a second row.
#pragma unroll
      for (int r = 0; r < I::template per<R>(); ++r)
#pragma unroll
        for (int j = 0; j < R; ++j) {
          const int b = tid + r * NT;
          if (!(E / R % NT == 0 || b < E / R)) continue;
          const long t = static_cast<long>(I::template input<R>(b) + j * (L / R)) * S + s0 +
                         I::template sequence<R>(b);
          u[r][j] = scale(-0.5 * P.absorber_rate[t], held[r][out_at<R>(j)]);
        }
      __syncthreads();
      transform_out(1);
    }
  } else {
    // At the bins: the transformed response and the absorber's term laid out in LDS, a
    // loop over the points, and the next stage's input in their place.
    __shared__ cplx second_row[Kind == kEntry ? 1 : E];
    if constexpr (Kind != kEntry) {
      transform_in(0);
      __syncthreads();
      I::outputs(w, [&](cplx& x, int s, int k) { lds[k * G + s] = x; });
      if (P.absorber_stream >= 0) {
        __syncthreads();
        I::outputs(w, [&](cplx& x, int s, int k) { second_row[k * G + s] = lds[k * G + s]; });
        __syncthreads();
        transform_in(1);
        __syncthreads();
        // Row 0 back in `lds`, row 1 in `second_row`.
        I::outputs(w, [&](cplx& x, int s, int k) {
          lds[k * G + s] = second_row[k * G + s];
          second_row[k * G + s] = x;
        });
      }
      __syncthreads();
    }
    [[maybe_unused]] double v0 = 0.0, v1 = 0.0, v2 = 0.0;
#pragma unroll 1
    for (int e = tid; e < E; e += NT) {
      if constexpr (POINTS > 1) ahead(e);
      if (bin < 0) {
        if constexpr (Kind != kAccept) lds[e] = make(0.0, 0.0);
        continue;
      }
      if constexpr (Kind != kEntry) {
        const cplx response = lds[e];
        const cplx absorber = finish.absorbed ? second_row[e] : make(0.0, 0.0);
        if constexpr (Kind == kFinish) {
          const cplx k = bin_derivative(a, finish, stage - 1, bin, response, absorber);
          entry.comb = add(entry.comb, scale(P.tab_a[stage * P.n_stages + stage - 1], k));
        } else {
          const cplx k = bin_derivative(a, finish, stage, bin, response, absorber);
          cplx sol = make(0.0, 0.0), err = make(0.0, 0.0);
          for (int i = 0; i < stage; ++i) {
            const cplx ki = a.k[static_cast<long>(i) * P.N + bin];
            sol = add(sol, scale(P.tab_b[i], ki));
            err = add(err, scale(P.tab_e[i], ki));
          }
          sol = add(sol, scale(P.tab_b[stage], k));
          err = add(err, scale(P.tab_e[stage], k));
          const cplx whole = cexp(phase_sum(a.R->whole.phi_w, P.phi, P.n_phi, P.N, bin));
          const cplx y = a.y[bin];
          const cplx yn = mul(whole, add(y, scale(a.R->dz, sol)));
          a.adv[bin] = yn;
          a.recycled[bin] = mul(whole, k);
          if (P.normmask[bin]) {
            v0 = v0 + norm2(y);
            v1 = v1 + norm2(yn);
            v2 = v2 + norm2(mul(whole, scale(a.R->dz, err)));
          }
        }
      }
      if constexpr (Kind != kAccept) lds[e] = bin_input(a, entry, bin);
    }
    if constexpr (Kind == kAccept) {
      // Three masked sums a workgroup, in a fixed order.
      __shared__ double sums[3][NT];
      sums[0][tid] = v0;
      sums[1][tid] = v1;
      sums[2][tid] = v2;
      __syncthreads();
      for (int half = NT / 2; half > 0; half >>= 1) {
        if (tid < half)
          for (int i = 0; i < 3; ++i) sums[i][tid] = sums[i][tid] + sums[i][tid + half];
        __syncthreads();
      }
      if (tid < 3)
        store_awaited(a.partials + tid * static_cast<int>(gridDim.x) + group, sums[tid][0]);
    } else {
      __syncthreads();
      F::inputs(u, [&](cplx& x, int s, int k) { x = lds[k * G + s]; });
      __syncthreads();
      transform_out(0);
    }
  }
}

// The damped Raman response as the T-point kernel w (h1 + i h2), the spacing folded in
// (its transform is the product's factor).
__global__ void raman_kernel_fill(DeviceProblem P, const TrialRecord* R, int stage,
                                  const cplx* twist, cplx* z) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= P.T) return;
  const long n2 = 2L * P.T;
  double h[2];
  for (int q = 0; q < 2; ++q) {
    const long m = t + static_cast<long>(q) * P.T;
    const double delay = static_cast<double>(m) * P.dt_fine;
    double total = 0.0;
    for (int r = 0; r < P.n_raman; ++r)
      total = total + P.raman_rows[r * n2 + m] * exp(-R->stage[stage].raman_rate[r] * delay);
    h[q] = P.raman_fraction * total * P.dt_fine;
  }
  z[t] = mul(twist[t], make(h[0], h[1]));
}

template <int LOG2L, int Kind>
void launch_kind(const EnvStage& a, int stage, hipStream_t s) {
  using H = EnvShape<LOG2L, Kind>;
  const unsigned blocks = static_cast<unsigned>((a.P.T >> LOG2L) / H::G);
  SP_CHECK(LOG2L < 8 || blocks % 8 == 0, "the groups of long sequences run in eights");
  hipLaunchKernelGGL((env_kernel<LOG2L, Kind>), dim3(blocks), dim3(H::THREADS), 0, s, a, stage);
}

template <int Kind>
void launch(const EnvStage& a, int log2l, int stage, hipStream_t s) {
  switch (log2l) {
    case 2: launch_kind<2, Kind>(a, stage, s); break;
    case 3: launch_kind<3, Kind>(a, stage, s); break;
    case 4: launch_kind<4, Kind>(a, stage, s); break;
    case 5: launch_kind<5, Kind>(a, stage, s); break;
    case 6: launch_kind<6, Kind>(a, stage, s); break;
    case 7: launch_kind<7, Kind>(a, stage, s); break;
    case 8: launch_kind<8, Kind>(a, stage, s); break;
    case 9: launch_kind<9, Kind>(a, stage, s); break;
    case 10: launch_kind<10, Kind>(a, stage, s); break;
    case 11: launch_kind<11, Kind>(a, stage, s); break;
    case 12: launch_kind<12, Kind>(a, stage, s); break;
    default: throw Error(kValue, "an envelope grid has 2^4 to 2^24 fine samples");
  }
  SP_HIP(hipGetLastError());
}

}  // namespace

unsigned env_accept_blocks(const EnvStage& a) {
  return static_cast<unsigned>((a.P.T >> a.log2n1) >> env_log2g(a.log2n1, true));
}

void launch_env_raman_kernel(const EnvStage& a, int stage, cplx* z, hipStream_t s) {
  hipLaunchKernelGGL(raman_kernel_fill, dim3(blocks_for(a.P.T, 256)), dim3(256), 0, s, a.P, a.R,
                     stage, a.twist, z);
  SP_HIP(hipGetLastError());
}

void launch_env_entry(const EnvStage& a, int stage, hipStream_t s) {
  launch<kEntry>(a, a.log2n1, stage, s);
}
void launch_env_drive(const EnvStage& a, int stage, hipStream_t s) {
  launch<kDrive>(a, a.log2n2, stage, s);
}
void launch_env_product(const EnvStage& a, int stage, hipStream_t s) {
  launch<kProduct>(a, a.log2n1, stage, s);
}
void launch_env_response(const EnvStage& a, int stage, hipStream_t s) {
  launch<kResponse>(a, a.log2n2, stage, s);
}
void launch_env_finish(const EnvStage& a, int stage, hipStream_t s) {
  launch<kFinish>(a, a.log2n1, stage, s);
}
void launch_env_accept(const EnvStage& a, hipStream_t s) {
  launch<kAccept>(a, a.log2n1, a.P.n_stages - 1, s);
}

}  // namespace sp
