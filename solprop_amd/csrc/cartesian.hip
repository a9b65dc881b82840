// The free-space Cartesian route (see cartesian.hpp).
#include "cartesian.hpp"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <string>

#include "fft_regs.hpp"
#include "sync.hpp"

namespace sp {
namespace {

struct KerrArgs {
  double coefficient, self, conj_term;
};

__device__ inline cplx kerr_point(cplx e, const KerrArgs& k) {
  cplx p = scale(k.self * norm2(e), e);
  if (k.conj_term != 0.0) p = add(p, scale(k.conj_term, mul(mul(e, e), conj(e))));
  return scale(k.coefficient, p);
}

// Every pass is bound by HBM: a volume does not fit the caches, so the passes' count of
// volume reads and writes sets the time, and each pass has to keep enough of them in
// flight. The transforms therefore run radix-16 stages in registers (fft_regs.hpp): a
// thread's 16 loads are issued together, and a 256-point sequence crosses LDS once.
// 256 x 128 x 512 points (268 MB a pass either way), before with radix-4 stages in LDS and
// now: x pass 158 -> 84 us (6.4 TB/s), y response 140 -> 98 us.

// A thread of a strided pass holds a radix-16 butterfly, or a whole sequence where that is
// shorter.
template <int LOG2L, int G, bool RestFirst>
using AxisFft = RegsFft<LOG2L, G, true, RestFirst, (LOG2L < 4 ? LOG2L : 4)>;

// The x axis: G neighbouring sequences (points `stride` apart, blocks of L stride points).
template <int LOG2L, int G, int Sign>
__global__ void __launch_bounds__((AxisFft<LOG2L, G, false>::NT))
    cart_x(cplx* f, long stride, const cplx* __restrict__ tw) {
  using F = AxisFft<LOG2L, G, false>;
  __shared__ cplx lds[F::LDS_POINTS];
  cplx* at = f + static_cast<long>(blockIdx.y) * F::L * stride + static_cast<long>(blockIdx.x) * G;
  typename F::First v;
  typename F::Last w;
  F::inputs(v, [&](cplx& x, int s, int j) { x = at[j * stride + s]; });
  F::run(v, w, lds, tw, Sign);
  F::outputs(w, [&](cplx& x, int s, int j) { at[j * stride + s] = x; });
}

// The y axis's inverse transform, the response at every point and the forward transform
// in one pass, in place: the forward transform's stages run in the reverse order of
// radices, so that it starts from the registers the inverse ends with.
template <int LOG2L, int G>
__global__ void __launch_bounds__((AxisFft<LOG2L, G, false>::NT))
    cart_y_response(cplx* f, long stride, const cplx* __restrict__ tw, KerrArgs k) {
  using I = AxisFft<LOG2L, G, false>;
  using F = AxisFft<LOG2L, G, true>;
  __shared__ cplx lds[I::LDS_POINTS];
  cplx* at = f + static_cast<long>(blockIdx.x) * G;
  typename I::First v;
  typename I::Last w;
  I::inputs(v, [&](cplx& x, int s, int j) { x = at[j * stride + s]; });
  I::run(v, w, lds, tw, +1);
  // Both transforms order a butterfly's points alike; the inverse leaves them permuted.
  typename F::First u;
  constexpr int R = F::radix(0);
#pragma unroll
  for (int r = 0; r < F::template per<R>(); ++r)
#pragma unroll
    for (int j = 0; j < R; ++j) u[r][j] = kerr_point(w[r][out_at<R>(j)], k);
  __syncthreads();  // the inverse's last hand-over is read
  typename F::Last z;
  F::run(u, z, lds, tw, -1);
  F::outputs(z, [&](cplx& x, int s, int j) { at[j * stride + s] = x; });
}

// The t axis (contiguous rows) and what happens to its spectrum between two source
// evaluations, so that the spectrum of a source and of the next stage's input are never
// stored: G rows of the field are transformed forward in registers, laid out in LDS, and
// a loop over the points applies the prefactor and the register pass of the low-storage
// step (J. Hult, J. Lightwave Technol. 25, 3770 (2007), in the reference's three-register
// form, src/solprop/backends/numpy_ref/engines.py:432-480): y the state A, acc the
// accumulator, prev the previous source (for the stiffness indicator). R[0].x_w and
// R[1].x_w weigh the operator to the middle and to the end. The next stage's input is
// transformed back in registers and stored as the field. The kinds:
//   kInverse  the spectrum `y` into the field (a step's first input)
//   kSource   the source alone into `acc`
//   kPass 1..3 forward, register pass, inverse; kPass 4 forward, register pass (the state).
// Passes 2 to 4 leave a masked sum per workgroup (|S2 - g|^2, |S3 - S2|^2, |A|^2), in a
// fixed order. On 256 x 128 x 512 points stages 1 to 4 take 325, 320, 376 and 242 us
// (4.4 to 5.4 TB/s), a step 2.44 ms (5.95 with the transforms and the passes apart and
// radix-4). A step moves 53 volumes, or 49.5 where the
// tables are imaginary (69 with the transforms and the passes apart).
enum TKind : int { kInverse = 0, kPass1, kPass2, kPass3, kPass4, kSource };

struct TArgs {
  cplx* f;
  cplx *y, *acc, *prev;
  const void* pref;  // a table of cplx, or with Imaginary of doubles (the imaginary parts)
  const void* phi;
  const unsigned char* scored;
  const AdamsRecord* R;
  double* sums;
};

// Imaginary: the operator and the prefactor have no real part (a lossless medium), and
// their tables hold the imaginary part alone, half the bytes; the products are the same.
template <bool Imaginary>
__device__ inline cplx table_times(const void* table, long idx, cplx v) {
  if constexpr (Imaginary) {
    const double b = static_cast<const double*>(table)[idx];
    return make(-(b * v.y), b * v.x);
  } else {
    return mul(static_cast<const cplx*>(table)[idx], v);
  }
}

template <bool Imaginary>
__device__ inline cplx table_flow(const void* table, long idx, double w) {
  if constexpr (Imaginary) {
    double sine, cosine;
    sincos(w * static_cast<const double*>(table)[idx], &sine, &cosine);
    return make(cosine, sine);
  } else {
    return cexp(scale(w, static_cast<const cplx*>(table)[idx]));
  }
}

template <int LOG2L, int G, int LOGR, int Kind, bool Imaginary>
__global__ void __launch_bounds__((RegsFft<LOG2L, G, false, false, LOGR>::NT))
    cart_t(TArgs a, const cplx* __restrict__ tw) {
  using F = RegsFft<LOG2L, G, false, false, LOGR>;
  constexpr int L = F::L, E = F::E, NT = F::NT;
  __shared__ cplx lds[F::LDS_POINTS];
  __shared__ double tree[NT];
  const long base = static_cast<long>(blockIdx.x) * E;
  const int tid = threadIdx.x;
  if constexpr (Kind != kInverse) {
    typename F::First v;
    typename F::Last w;
    F::inputs(v, [&](cplx& x, int s, int j) { x = a.f[base + s * L + j]; });
    F::run(v, w, lds, tw, -1);
    __syncthreads();  // the last hand-over is read
    F::outputs(w, [&](cplx& x, int s, int j) { lds[F::slot(s, j)] = x; });
    __syncthreads();
    double sq = 0.0;
    const double h = a.R[0].dz;
    const double flow_w = a.R[Kind == kPass1 ? 0 : 1].x_w[0];
#pragma unroll 2
    for (int e = tid; e < E; e += NT) {
      const long idx = base + e;
      cplx& slot = lds[F::slot(e / L, e % L)];
      const cplx s = table_times<Imaginary>(a.pref, idx, slot);
      const bool scored = Kind != kSource && a.scored[e % L] != 0;
      if constexpr (Kind == kSource) {
        a.acc[idx] = s;
      } else if constexpr (Kind == kPass1) {
        const cplx flow = table_flow<Imaginary>(a.phi, idx, flow_w);
        const cplx state = mul(flow, a.y[idx]);
        const cplx g = mul(flow, s);
        a.y[idx] = state;
        a.prev[idx] = g;
        slot = add(state, scale(0.5 * h, g));
      } else if constexpr (Kind == kPass2) {
        const cplx g = a.prev[idx], state = a.y[idx];
        const cplx d = sub(s, g);
        if (scored) sq += norm2(d);
        a.acc[idx] = add(add(state, scale(h / 6.0, g)), scale(h / 3.0, s));
        a.prev[idx] = s;
        slot = add(state, scale(0.5 * h, s));
      } else if constexpr (Kind == kPass3) {
        const cplx d = sub(s, a.prev[idx]);
        if (scored) sq += norm2(d);
        a.acc[idx] = add(a.acc[idx], scale(h / 3.0, s));
        const cplx flow = table_flow<Imaginary>(a.phi, idx, flow_w);
        slot = mul(flow, add(a.y[idx], scale(h, s)));
      } else {
        const cplx flow = table_flow<Imaginary>(a.phi, idx, flow_w);
        const cplx state = add(mul(flow, a.acc[idx]), scale(h / 6.0, s));
        a.y[idx] = state;
        if (scored) sq += norm2(state);
      }
    }
    if constexpr (Kind >= kPass2 && Kind <= kPass4) {
      tree[tid] = sq;
      __syncthreads();
      for (int half = NT / 2; half > 0; half /= 2) {
        if (tid < half) tree[tid] = tree[tid] + tree[tid + half];
        __syncthreads();
      }
      if (tid == 0) a.sums[static_cast<long>(Kind - kPass2) * gridDim.x + blockIdx.x] = tree[0];
    }
  }
  if constexpr (Kind <= kPass3) {
    typename F::First v;
    typename F::Last w;
    if constexpr (Kind == kInverse) {
      F::inputs(v, [&](cplx& x, int s, int j) { x = a.y[base + s * L + j]; });
    } else {
      __syncthreads();
      F::inputs(v, [&](cplx& x, int s, int j) { x = lds[F::slot(s, j)]; });
      __syncthreads();
    }
    F::run(v, w, lds, tw, +1);
    F::outputs(w, [&](cplx& x, int s, int j) { a.f[base + s * L + j] = x; });
  }
}

__global__ void find_real_part(const cplx* __restrict__ table, std::size_t n, int* found) {
  bool any = false;
  for (std::size_t i = static_cast<std::size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<std::size_t>(gridDim.x) * blockDim.x)
    any = any || !(table[i].x == 0.0);
  if (any) *found = 1;
}

__global__ void take_imaginary(const cplx* __restrict__ table, std::size_t n,
                               double* __restrict__ out) {
  for (std::size_t i = static_cast<std::size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<std::size_t>(gridDim.x) * blockDim.x)
    out[i] = table[i].y;
}

template <int LOG2L, int G>
struct XPass {
  static void launch(dim3 grid, hipStream_t s, cplx* f, long stride, const cplx* tw, int sign) {
    constexpr int NT = AxisFft<LOG2L, G, false>::NT;
    if (sign > 0)
      hipLaunchKernelGGL((cart_x<LOG2L, G, 1>), grid, dim3(NT), 0, s, f, stride, tw);
    else
      hipLaunchKernelGGL((cart_x<LOG2L, G, -1>), grid, dim3(NT), 0, s, f, stride, tw);
  }
};

template <int LOG2L, int G>
struct YResponse {
  static void launch(unsigned blocks, hipStream_t s, cplx* f, long stride, const cplx* tw,
                     KerrArgs k) {
    hipLaunchKernelGGL((cart_y_response<LOG2L, G>), dim3(blocks),
                       dim3(AxisFft<LOG2L, G, false>::NT), 0, s, f, stride, tw, k);
  }
};

template <int LOG2L, int G, int LOGR>
struct TStage {
  template <bool Imaginary>
  static void launch(int kind, unsigned blocks, hipStream_t s, const TArgs& a, const cplx* tw) {
    const dim3 grid(blocks), block(RegsFft<LOG2L, G, false, false, LOGR>::NT);
    switch (kind) {
      case kInverse:  // reads neither table
        hipLaunchKernelGGL((cart_t<LOG2L, G, LOGR, kInverse, true>), grid, block, 0, s, a, tw);
        break;
      case kPass1:
        hipLaunchKernelGGL((cart_t<LOG2L, G, LOGR, kPass1, Imaginary>), grid, block, 0, s, a, tw);
        break;
      case kPass2:
        hipLaunchKernelGGL((cart_t<LOG2L, G, LOGR, kPass2, Imaginary>), grid, block, 0, s, a, tw);
        break;
      case kPass3:
        hipLaunchKernelGGL((cart_t<LOG2L, G, LOGR, kPass3, Imaginary>), grid, block, 0, s, a, tw);
        break;
      case kPass4:
        hipLaunchKernelGGL((cart_t<LOG2L, G, LOGR, kPass4, Imaginary>), grid, block, 0, s, a, tw);
        break;
      default:
        hipLaunchKernelGGL((cart_t<LOG2L, G, LOGR, kSource, Imaginary>), grid, block, 0, s, a, tw);
    }
  }
};

// The strided passes' shapes: workgroups of at most kMaxElems points, 16 sequences or, on an
// axis of at most kShortAxis points, 64 (a thread each).
constexpr int kShortAxis = 8;

template <template <int, int> class Op, int LOG2L, typename... A>
void dispatch_g(int log2g, A... a) {
  constexpr int L = 1 << LOG2L;
  switch (log2g) {
    case 0: Op<LOG2L, 1>::launch(a...); return;
    case 1: if constexpr (L * 2 <= kMaxElems) { Op<LOG2L, 2>::launch(a...); return; } break;
    case 2: if constexpr (L * 4 <= kMaxElems) { Op<LOG2L, 4>::launch(a...); return; } break;
    case 3: if constexpr (L * 8 <= kMaxElems) { Op<LOG2L, 8>::launch(a...); return; } break;
    case 4: if constexpr (L * 16 <= kMaxElems) { Op<LOG2L, 16>::launch(a...); return; } break;
    case 5: if constexpr (L <= kShortAxis) { Op<LOG2L, 32>::launch(a...); return; } break;
    case 6: if constexpr (L <= kShortAxis) { Op<LOG2L, 64>::launch(a...); return; } break;
    default: break;
  }
  throw Error(kValue, "no Cartesian pass kernel for this shape");
}

template <template <int, int> class Op, typename... A>
void dispatch(int log2l, int log2g, A... a) {
  switch (log2l) {
    case 2: dispatch_g<Op, 2>(log2g, a...); break;
    case 3: dispatch_g<Op, 3>(log2g, a...); break;
    case 4: dispatch_g<Op, 4>(log2g, a...); break;
    case 5: dispatch_g<Op, 5>(log2g, a...); break;
    case 6: dispatch_g<Op, 6>(log2g, a...); break;
    case 7: dispatch_g<Op, 7>(log2g, a...); break;
    case 8: dispatch_g<Op, 8>(log2g, a...); break;
    case 9: dispatch_g<Op, 9>(log2g, a...); break;
    case 10: dispatch_g<Op, 10>(log2g, a...); break;
    case 11: dispatch_g<Op, 11>(log2g, a...); break;
    case 12: dispatch_g<Op, 12>(log2g, a...); break;
    default: throw Error(kValue, "a Cartesian axis has 4 to 4096 points");
  }
  SP_HIP(hipGetLastError());
}

// The t rows a workgroup owns (log2): enough for 2^10 points (one wave of 16 points a
// thread, so that its barriers wait for nobody: stage 1 344 -> 325 us and stage 4 265 ->
// 242 us against 2^11 points on 512-point rows). Where that leaves fewer than 1024
// workgroups the chip is not full and a step waits for one thread's chain of points: then
// 2^8 points and four a thread (16 a thread are a quarter of a wave and as long a chain),
// up to rows of 2048 points; 4096 are 256 threads either way and 5 % faster at 16 points.
// A step on 16 x 32 x 256 points: 104 us, 136-167 at 16 points a thread. Narrow and wide
// on 64 x 64 x 64 (256 wide workgroups) 125 and 137 us, on 128 x 128 x 64 (1024) 253 and
// 259, on 64 x 64 x 512 (2048) 384 and 351. At most 16 rows, which divide any grid's nx ny.
constexpr int t_log2g(int log2l, bool wide) {
  const int g = (wide ? 10 : 8) - log2l;
  return g < 0 ? 0 : (g > 4 ? 4 : g);
}

constexpr int t_logr(int log2l, bool wide) { return wide || log2l > 11 ? 4 : 2; }

template <int LOG2L>
void dispatch_t_wide(bool wide, bool imaginary, int kind, long rows, hipStream_t s,
                     const TArgs& a, const cplx* tw) {
  constexpr int W = t_log2g(LOG2L, true), N = t_log2g(LOG2L, false);
  using Wide = TStage<LOG2L, (1 << W), t_logr(LOG2L, true)>;
  using Narrow = TStage<LOG2L, (1 << N), t_logr(LOG2L, false)>;
  // A narrow workgroup fills a wave (but on rows of 4 and 8 points, 16 rows at most).
  static_assert(RegsFft<LOG2L, (1 << N), false, false, t_logr(LOG2L, false)>::NT >=
                (LOG2L < 4 ? 4 << LOG2L : 64));
  const unsigned blocks = static_cast<unsigned>(rows >> (wide ? W : N));
  if (wide && imaginary)
    Wide::template launch<true>(kind, blocks, s, a, tw);
  else if (wide)
    Wide::template launch<false>(kind, blocks, s, a, tw);
  else if (imaginary)
    Narrow::template launch<true>(kind, blocks, s, a, tw);
  else
    Narrow::template launch<false>(kind, blocks, s, a, tw);
}

void dispatch_t(int log2l, bool wide, bool imaginary, int kind, long rows, hipStream_t s,
                const TArgs& a, const cplx* tw) {
  switch (log2l) {
    case 2: dispatch_t_wide<2>(wide, imaginary, kind, rows, s, a, tw); break;
    case 3: dispatch_t_wide<3>(wide, imaginary, kind, rows, s, a, tw); break;
    case 4: dispatch_t_wide<4>(wide, imaginary, kind, rows, s, a, tw); break;
    case 5: dispatch_t_wide<5>(wide, imaginary, kind, rows, s, a, tw); break;
    case 6: dispatch_t_wide<6>(wide, imaginary, kind, rows, s, a, tw); break;
    case 7: dispatch_t_wide<7>(wide, imaginary, kind, rows, s, a, tw); break;
    case 8: dispatch_t_wide<8>(wide, imaginary, kind, rows, s, a, tw); break;
    case 9: dispatch_t_wide<9>(wide, imaginary, kind, rows, s, a, tw); break;
    case 10: dispatch_t_wide<10>(wide, imaginary, kind, rows, s, a, tw); break;
    case 11: dispatch_t_wide<11>(wide, imaginary, kind, rows, s, a, tw); break;
    case 12: dispatch_t_wide<12>(wide, imaginary, kind, rows, s, a, tw); break;
    default: throw Error(kValue, "a Cartesian axis has 4 to 4096 points");
  }
  SP_HIP(hipGetLastError());
}

int log2_of(int n) {
  int m = 0;
  while ((1 << m) < n) ++m;
  return m;
}

// Sequences (log2) a workgroup of a strided pass owns, of `count` neighbouring ones in each
// of `blocks` blocks: runs of up to 16 points, never more than `max_points` points in all.
// A short axis takes a wave of sequences where 256 workgroups remain: at 16 sequences of 8
// points the y pass on 32 x 8 x 2048 ran workgroups of 8 threads and took 21 us, 7.4 in
// LDS before. (16 points are 16 threads' butterflies and take what they took, 13.6 us on
// 256 x 16 x 512.)
int axis_log2g(int n, long count, long blocks, int max_points) {
  int g = 0;
  const int cap = std::min(max_points, kMaxElems), most = n <= kShortAxis ? 6 : 4;
  while (g < most && n * (1 << (g + 1)) <= cap && count % (1L << (g + 1)) == 0 &&
         (g < 4 || (count >> (g + 1)) * blocks >= 256))
    ++g;
  return g;
}

enum Phase : int { kUpload, kPassT, kPassX, kPassY, kLs1, kLs2, kLs3, kLs4, kNorms };
const char* const kPhaseNames[] = {"record upload", "t inverse", "x pass", "y response",
                                   "t stage 1", "t stage 2", "t stage 3", "t stage 4",
                                   "norms"};

struct ReplayEngine final : march::Engine {
  std::function<double(double, double)> step;
  std::function<void(double)> commit;
  double trial(double z, double dz) override { return step(z, dz); }
  void accept(double dz) override { commit(dz); }
};

struct ReplayHost final : march::Host {
  AttemptLog& log;
  explicit ReplayHost(AttemptLog& l) : log(l) {}
  void record(double end, double dz, double norm, bool acc) override {
    log.record(end, dz, norm, acc);
  }
  bool halt() override { return log.halt(); }
};

}  // namespace

template <typename T>
T* CartesianWorkspace::alloc(std::size_t n) {
  T* p = nullptr;
  if (n == 0) n = 1;
  SP_HIP(hipMalloc(&p, n * sizeof(T)));
  allocations_.push_back(p);
  device_bytes_ += n * sizeof(T);
  return p;
}

CartesianWorkspace::CartesianWorkspace(const sp_problem_desc& d) {
  // Refusals first, before anything is allocated.
  SP_CHECK(d.kind == 2, "the Cartesian workspace runs the free-space (x, y, t) grid");
  SP_CHECK(d.method == 2 && d.n_schedule >= 1 && d.schedule_edges,
           "the Cartesian route runs the low-storage RK4IP replay of a schedule");
  nx_ = d.grid_nx;
  ny_ = d.grid_ny;
  nt_ = d.n_omega;
  auto pow2 = [](int v, int lo, int hi) { return v >= lo && v <= hi && (v & (v - 1)) == 0; };
  SP_CHECK(pow2(nx_, 4, 4096) && pow2(ny_, 4, 4096) && pow2(nt_, 4, 4096),
           "the Cartesian grid's nx, ny and nt are powers of two from 4 to 4096");
  SP_CHECK(d.n_modes == nx_ * ny_, "a Cartesian grid's columns are its nx ny points");
  SP_CHECK(d.n_t == nt_ && d.n_to == nt_, "a Cartesian grid's time axis is n_t = n_to");
  SP_CHECK(d.n_phi == 1 && d.phi_terms, "the Cartesian route's operator is one constant table");
  SP_CHECK(d.n_prefactor == 1 && d.prefactor_terms, "one constant prefactor table");
  SP_CHECK(!d.has_plasma && d.n_raman == 0 && d.absorber_scheme == 0 && !d.spatial_absorber,
           "the Cartesian route is built with the Kerr response alone");
  SP_CHECK(d.has_kerr == 0 || d.kerr_real == 0, "the Cartesian envelope takes the analytic Kerr form");
  SP_CHECK(d.phi_paths[0].kind == 1, "the Cartesian operator's weight is W(z) = z");
  SP_CHECK(d.prefactor_paths[0].kind == 0 && d.density.kind == 0,
           "the Cartesian prefactor and density are constant");
  for (int i = 0; i < d.n_schedule; ++i)
    SP_CHECK(d.schedule_edges[i + 1] > d.schedule_edges[i], "the schedule's edges must increase");
  V_ = static_cast<std::size_t>(nx_) * ny_ * nt_;
  SP_CHECK(V_ <= (std::size_t{1} << 31), "the volume holds at most 2^31 samples");
  edges_.assign(d.schedule_edges, d.schedule_edges + d.n_schedule + 1);
  for (int i = 0; i < d.n_schedule; ++i) steps_.push_back(edges_[i + 1] - edges_[i]);
  const double v = static_cast<double>(V_);
  kerr_self_ = d.has_kerr ? d.kerr_self : 0.0;
  kerr_conj_ = d.has_kerr ? d.kerr_conjugate : 0.0;
  // gamma = the Kerr coefficient times the density times the prefactor's constant weight.
  kerr_scale_ = d.has_kerr ? d.kerr_coefficient * d.density.value * d.prefactor_paths[0].value /
                                 (v * v * v)
                           : 0.0;
  const char* env = std::getenv("SOLPROP_MI355X_GRAPH");
  use_graphs_ = !(env && env[0] == '0');
  // The strided passes' workgroup tile, points (a launch shape only: every sequence's
  // arithmetic is the same whichever is chosen).
  const char* tile = std::getenv("SOLPROP_MI355X_CARTESIAN_TILE");
  const int max_points = tile ? std::atoi(tile) : 4096;
  SP_CHECK(max_points >= 4 && max_points <= 4096,
           "SOLPROP_MI355X_CARTESIAN_TILE is 4 to 4096 points");
  const long rows = static_cast<long>(nx_) * ny_;
  const int lt = log2_of(nt_);
  wide_t_ = (rows >> t_log2g(lt, true)) >= 1024;
  t_blocks_ = static_cast<int>(rows >> t_log2g(lt, wide_t_));
  gx_ = axis_log2g(nx_, nt_, ny_, max_points);
  gy_ = axis_log2g(ny_, static_cast<long>(nx_) * nt_, 1, max_points);
  try {
    SP_HIP(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking));
    const int C = nx_ * ny_, N = nt_;
    P_.kind = 2;
    P_.C = C;
    P_.N = N;
    P_.T = N;
    P_.NF = N;
    P_.n_phi = 1;
    P_.n_pref = 1;
    P_.Q = 1;
    std::vector<unsigned char> ones(static_cast<std::size_t>(N), 1);
    auto* active = alloc<unsigned char>(N);
    SP_HIP(hipMemcpy(active, ones.data(), N, hipMemcpyHostToDevice));
    P_.active = active;
    auto* nm = alloc<unsigned char>(N);
    SP_HIP(hipMemcpy(nm, d.norm_mask, N, hipMemcpyHostToDevice));
    P_.normmask = nm;
    B_.y = alloc<cplx>(V_);
    B_.advanced = alloc<cplx>(V_);
    field_ = alloc<cplx>(V_);
    acc_ = alloc<cplx>(V_);
    prev_ = alloc<cplx>(V_);
    save_ = alloc<cplx>(V_);
    // The tables' layout is decided, and the imaginary parts taken, on the device.
    auto* real_part = alloc<int>(1);
    SP_HIP(hipMemcpy(save_, d.phi_terms, V_ * sizeof(cplx), hipMemcpyHostToDevice));
    SP_HIP(hipMemcpy(field_, d.prefactor_terms, V_ * sizeof(cplx), hipMemcpyHostToDevice));
    SP_HIP(hipMemsetAsync(real_part, 0, sizeof(int), stream_));
    const dim3 grid(4096), block(256);
    hipLaunchKernelGGL(find_real_part, grid, block, 0, stream_, save_, V_, real_part);
    hipLaunchKernelGGL(find_real_part, grid, block, 0, stream_, field_, V_, real_part);
    SP_HIP(hipGetLastError());
    int found = 0;
    SP_HIP(hipStreamSynchronize(stream_));
    SP_HIP(hipMemcpy(&found, real_part, sizeof(int), hipMemcpyDeviceToHost));
    imaginary_ = found == 0;
    auto table = [&](const cplx* src) -> const void* {
      if (imaginary_) {
        auto* p = alloc<double>(V_);
        hipLaunchKernelGGL(take_imaginary, grid, block, 0, stream_, src, V_, p);
        SP_HIP(hipGetLastError());
        return p;
      }
      auto* p = alloc<cplx>(V_);
      SP_HIP(hipMemcpyAsync(p, src, V_ * sizeof(cplx), hipMemcpyDeviceToDevice, stream_));
      return p;
    };
    phi_ = table(save_);
    pref_ = table(field_);
    SP_HIP(hipStreamSynchronize(stream_));
    auto roots = [&](int n) {
      const auto host = unit_roots(static_cast<std::size_t>(n));
      auto* p = alloc<cplx>(host.size());
      SP_HIP(hipMemcpy(p, host.data(), host.size() * sizeof(cplx), hipMemcpyHostToDevice));
      return p;
    };
    roots_t_ = roots(nt_);
    roots_x_ = roots(nx_);
    roots_y_ = roots(ny_);
    rec_dev_ = alloc<AdamsRecord>(3);
    SP_HIP(hipHostMalloc(reinterpret_cast<void**>(&rec_host_), 3 * sizeof(AdamsRecord)));
    std::memset(rec_host_, 0, 3 * sizeof(AdamsRecord));
    partials_ = alloc<double>(ls_partials(static_cast<unsigned>(t_blocks_)));
    SP_HIP(hipHostMalloc(reinterpret_cast<void**>(&norms_host_), 4 * sizeof(double),
                         hipHostMallocMapped));
    SP_HIP(hipHostGetDevicePointer(reinterpret_cast<void**>(&B_.norms), norms_host_, 0));
    SP_HIP(hipEventCreateWithFlags(&done_, hipEventDisableTiming));
    events_.assign(kMarks, nullptr);
    for (auto& e : events_) SP_HIP(hipEventCreate(&e));
  } catch (...) {
    release();
    throw;
  }
}

CartesianWorkspace::~CartesianWorkspace() { release(); }

void CartesianWorkspace::release() {
  if (stream_) (void)hipStreamSynchronize(stream_);
  if (graph_) (void)hipGraphExecDestroy(graph_);
  graph_ = nullptr;
  for (void* p : allocations_) (void)hipFree(p);
  allocations_.clear();
  if (rec_host_) (void)hipHostFree(rec_host_);
  rec_host_ = nullptr;
  if (norms_host_) (void)hipHostFree(norms_host_);
  norms_host_ = nullptr;
  if (done_) (void)hipEventDestroy(done_);
  done_ = nullptr;
  for (auto& e : events_)
    if (e) (void)hipEventDestroy(e);
  events_.clear();
  if (stream_) (void)hipStreamDestroy(stream_);
  stream_ = nullptr;
}

void CartesianWorkspace::mark(int phase) {
  if (!marking_) return;
  const std::size_t k = marked_.size() + 1;
  SP_CHECK(k < events_.size(), "a profiled trial records at most 63 launches");
  SP_HIP(hipEventRecord(events_[k], stream_));
  marked_.push_back(phase);
}

void CartesianWorkspace::collect() {
  for (std::size_t k = 0; k < marked_.size(); ++k) {
    float ms = 0.0f;
    SP_HIP(hipEventElapsedTime(&ms, events_[k], events_[k + 1]));
    phase_ms_[marked_[k]] += ms;
    phase_n_[marked_[k]] += 1;
  }
  float total = 0.0f;
  if (!marked_.empty()) SP_HIP(hipEventElapsedTime(&total, events_[0], events_[marked_.size()]));
  trial_ms_ += total;
  timed_ += 1;
  marked_.clear();
}

std::vector<std::pair<const char*, double>> CartesianWorkspace::phases() const {
  std::vector<std::pair<const char*, double>> out;
  for (int i = 0; i < kPhases; ++i)
    if (phase_n_[i] > 0) out.emplace_back(kPhaseNames[i], phase_ms_[i] * 1e3 / phase_n_[i]);
  return out;
}

void CartesianWorkspace::enqueue_t(int kind, int phase) {
  const TArgs a{field_, B_.y, acc_, prev_, pref_, phi_, P_.normmask, rec_dev_, partials_};
  dispatch_t(log2_of(nt_), wide_t_, imaginary_, kind, static_cast<long>(nx_) * ny_, stream_, a, roots_t_);
  mark(phase);
}

// The transverse axes of a source evaluation, on the field the t rows' inverse left:
// x, then y with the response between its inverse and forward transforms, then x.
// Columns are iy nx + ix: the x axis has stride nt within each of ny blocks, the y axis
// stride nx nt.
void CartesianWorkspace::enqueue_transverse() {
  const long y_seqs = static_cast<long>(nx_) * nt_;
  const KerrArgs k{kerr_scale_, kerr_self_, kerr_conj_};
  const dim3 x_grid(static_cast<unsigned>(nt_ >> gx_), static_cast<unsigned>(ny_));
  const int lx = log2_of(nx_);
  dispatch<XPass>(lx, gx_, x_grid, stream_, field_, static_cast<long>(nt_),
                  static_cast<const cplx*>(roots_x_), +1);
  mark(kPassX);
  dispatch<YResponse>(log2_of(ny_), gy_, static_cast<unsigned>(y_seqs >> gy_), stream_, field_,
                      y_seqs, static_cast<const cplx*>(roots_y_), k);
  mark(kPassY);
  dispatch<XPass>(lx, gx_, x_grid, stream_, field_, static_cast<long>(nt_),
                  static_cast<const cplx*>(roots_x_), -1);
  mark(kPassX);
}

void CartesianWorkspace::enqueue_step() {
  if (marking_) SP_HIP(hipEventRecord(events_[0], stream_));
  SP_HIP(hipMemcpyAsync(rec_dev_, rec_host_, 3 * sizeof(AdamsRecord), hipMemcpyHostToDevice,
                        stream_));
  mark(kUpload);
  enqueue_t(kInverse, kPassT);
  for (int pass = 0; pass < 4; ++pass) {
    enqueue_transverse();
    enqueue_t(kPass1 + pass, kLs1 + pass);
  }
  launch_ls_norms(static_cast<unsigned>(t_blocks_), partials_, B_.norms, stream_);
  mark(kNorms);
}

void CartesianWorkspace::wait() {
  SP_HIP(hipEventRecord(done_, stream_));
  wait_event(done_);
}

double CartesianWorkspace::trial(double z, double dz) {
  // The constant operator's increments are the distances: Phi(z_m) - Phi(z) = z_m - z and
  // Phi(z + h) - Phi(z_m) = z + h - z_m, times the one table.
  const double mid = z + 0.5 * dz, end = z + dz;
  rec_host_[0].dz = dz;
  rec_host_[0].x_w[0] = mid - z;
  rec_host_[1].x_w[0] = end - mid;
  if (profile_) {
    marking_ = true;
    marked_.clear();
    try {
      enqueue_step();
    } catch (...) {
      marking_ = false;
      throw;
    }
    marking_ = false;
    wait();
    collect();
  } else if (use_graphs_) {
    if (!graph_) graph_ = capture_graph(stream_, [&] { enqueue_step(); });
    SP_HIP(hipGraphLaunch(graph_, stream_));
    graph_launches_ += 1;
    wait();
  } else {
    enqueue_step();
    wait();
  }
  trials_ += 1;
  evaluations_ += 4;
  const double lower = std::sqrt(norms_host_[0]), upper = std::sqrt(norms_host_[1]);
  stiffness_ = lower > 0.0 ? 2.0 * upper / lower : std::nan("");
  const double squared = norms_host_[2];
  return std::isfinite(squared) ? 0.0 : squared;
}

void CartesianWorkspace::load(double z, const double* field) {
  SP_CHECK(field != nullptr, "load needs a field");
  long cursor = -1;
  for (std::size_t i = 0; i < edges_.size(); ++i)
    if (march::reached(z, edges_[i]) && march::reached(edges_[i], z)) cursor = static_cast<long>(i);
  SP_CHECK(cursor >= 0, "a replay loads its state at one of its schedule's edges");
  transfer_.upload(B_.y, field, V_ * sizeof(cplx), stream_);
  state_ = march::State{};
  state_.z = edges_[static_cast<std::size_t>(cursor)];
  state_.cursor = cursor;
  loaded_ = true;
}

double CartesianWorkspace::probe_trial(double z, double dz) {
  if (!loaded_) throw Error(kState, "load a state before taking a trial");
  SP_HIP(hipMemcpyAsync(save_, B_.y, V_ * sizeof(cplx), hipMemcpyDeviceToDevice, stream_));
  const double norm = trial(z, dz);
  SP_HIP(hipMemcpyAsync(B_.advanced, B_.y, V_ * sizeof(cplx), hipMemcpyDeviceToDevice, stream_));
  SP_HIP(hipMemcpyAsync(B_.y, save_, V_ * sizeof(cplx), hipMemcpyDeviceToDevice, stream_));
  SP_HIP(hipStreamSynchronize(stream_));
  return norm;
}

void CartesianWorkspace::read_trial(double* out) {
  transfer_.download(out, B_.advanced, V_ * sizeof(cplx), stream_);
}

void CartesianWorkspace::read_state(double* out) {
  if (!loaded_) throw Error(kState, "no state is loaded");
  transfer_.download(out, B_.y, V_ * sizeof(cplx), stream_);
}

void CartesianWorkspace::export_state(const double* weight, bool optics, double* out) {
  read_state(out);
  const long n = static_cast<long>(V_);
  for (long i = 0; i < n; ++i) {
    double re = out[2 * i], im = out[2 * i + 1];
    if (weight) {
      const double s = std::sqrt(weight[i]);
      re = re * s;
      im = im * s;
    }
    if (optics) {
      im = -im;
      if ((i % nt_) & 1) {
        re = -re;
        im = -im;
      }
    }
    out[2 * i] = re;
    out[2 * i + 1] = im;
  }
}

bool CartesianWorkspace::advance_bounded(const Bounds& b, int columns, std::vector<double>& rows,
                                         sp_march_result* r) {
  if (!loaded_) throw Error(kState, "load a state before advancing");
  ReplayEngine engine;
  engine.step = [this](double z, double dz) { return trial(z, dz); };
  engine.commit = [this](double) { accepted_ += 1; };
  AttemptLog log;
  log.begin(&rows, columns, b);
  log.order = 4;
  ReplayHost host(log);
  const double target = std::min(b.target, edges_.back());
  bool done = false;
  try {
    done = march::replay_to(engine, host, state_, steps_, edges_, target) &&
           march::reached(state_.z, target);
  } catch (...) {
    r->z = state_.z;
    r->attempts = log.attempts;
    r->accepted = log.accepted;
    r->evaluations = evaluations_;
    throw;
  }
  r->z = state_.z;
  r->proposal = state_.cursor < static_cast<long>(steps_.size())
                    ? steps_[static_cast<std::size_t>(state_.cursor)]
                    : 0.0;
  r->done = done ? 1 : 0;
  r->attempts = log.attempts;
  r->accepted = log.accepted;
  r->evaluations = evaluations_;
  return done;
}

sp_counters CartesianWorkspace::counters() const {
  sp_counters c{};
  c.trials = trials_;
  c.evaluations = evaluations_;
  c.accepted = accepted_;
  c.graph_launches = graph_launches_;
  c.device_bytes = static_cast<long>(device_bytes_);
  return c;
}

std::vector<double> CartesianWorkspace::statistics(std::uint64_t, const double*, int,
                                                   const StatExtras&) {
  throw std::invalid_argument("plane statistics are not built on the Cartesian route");
}

void CartesianWorkspace::bind_monitor(const double*, const double*) {
  throw std::invalid_argument("the boundary monitor is not built on the Cartesian route");
}

void CartesianWorkspace::monitor_reading(double*) {
  throw std::invalid_argument("the boundary monitor is not built on the Cartesian route");
}

void CartesianWorkspace::source(double z, const double* lab, double* out, double* streams,
                                double* modal) {
  (void)z;
  SP_CHECK(lab && out && !streams && !modal, "the Cartesian source takes a spectrum and an output");
  SP_HIP(hipStreamSynchronize(stream_));
  // The state is kept: the spectrum takes its place for the inverse transform only.
  SP_HIP(hipMemcpy(save_, B_.y, V_ * sizeof(cplx), hipMemcpyDeviceToDevice));
  SP_HIP(hipMemcpy(B_.y, lab, V_ * sizeof(cplx), hipMemcpyHostToDevice));
  enqueue_t(kInverse, kPassT);
  SP_HIP(hipMemcpyAsync(B_.y, save_, V_ * sizeof(cplx), hipMemcpyDeviceToDevice, stream_));
  enqueue_transverse();
  enqueue_t(kSource, kLs1);
  SP_HIP(hipStreamSynchronize(stream_));
  SP_HIP(hipMemcpy(out, acc_, V_ * sizeof(cplx), hipMemcpyDeviceToHost));
}

long CartesianWorkspace::buffer(const char* name, double* out, long count) {
  SP_CHECK(name != nullptr, "a buffer name is required");
  if (std::strcmp(name, "stiffness") == 0) {
    if (out && count > 0) out[0] = stiffness_;
    return 1;
  }
  throw std::invalid_argument(std::string("no buffer named ") + name + " on the Cartesian route");
}

}  // namespace sp
