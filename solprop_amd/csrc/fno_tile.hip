// The surrogate's fused tile path (see fno_tile.hpp).
//
// What bounds it: the activations' traffic. A layer reads and writes (B, n, 64) BF16
// once in each direction (17 MB each way at 64 samples of 2048 bins); its products
// (1.6 GFLOP) take the matrix cores 2 us. Fragment layouts (v_mfma_f32_16x16x32_bf16): lane
// l holds row l % 16 of A, column l % 16 of B, elements 8 (l / 16) .. + 7 of K, and rows
// 4 (l / 16) .. + 3 of column l % 16 of the result. Activations are stored bin-major with
// the channels contiguous, so that a fragment contracting over channels is one 16-byte
// load straight from memory; the contraction over bins takes its tile from LDS, where the
// producing waves have just written it channel-major.
//
// Measured at the surrogate's shape (64 channels, 64 modes, 4 layers, 128 head units, 2048
// bins, 64 samples) against the general products of fno.hip, which write every
// pre-activation and gradient in FP32 and sum channels a workgroup each: a training step
// 4.43 ms -> 0.52 ms, a forward pass 0.92 ms -> 0.18 ms; a layer forward 26 us (1.3 TB/s of
// activations; the tile's load, contraction and hand-over in turn), backward 47 us.
#include "fno_tile.hpp"

#include <algorithm>

namespace sp::fno {
namespace {

typedef __bf16 v8b __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef unsigned short us8 __attribute__((ext_vector_type(8)));

constexpr float kGeluC = 0.7978845608028654f;  // sqrt(2 / pi)
constexpr float kGeluA = 0.044715f;
constexpr int kRow = kTile + 8;  // an LDS row of a tile's bins (16-byte rows, banks spread)

// LDS tiles are read 16 bytes a lane and written 8: the arrays start, and their rows lie,
// on 16-byte lines.
constexpr int kWide = 16;
template <typename T>
constexpr bool wide_pitch(int elements) {
  return elements * sizeof(T) % kWide == 0;
}
static_assert(wide_pitch<bf16>(kRow));

__device__ inline v8b load8(const bf16* p) { return *reinterpret_cast<const v8b*>(p); }

__device__ inline bf16 bf(float x) {
  return __builtin_bit_cast(bf16, static_cast<__bf16>(x));
}

__device__ inline uint2 bf4(float a, float b, float c, float d) {
  return make_uint2(static_cast<unsigned>(bf(a)) | static_cast<unsigned>(bf(b)) << 16,
                    static_cast<unsigned>(bf(c)) | static_cast<unsigned>(bf(d)) << 16);
}

__device__ inline v4f mfma(v8b a, v8b b, v4f c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ inline v4f mfma32(float a, float b, v4f c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// The tanh form of gelu by its smaller tail q = 1 / (1 + e^{2|u|}), u = c (x + a x^3):
// (1 + tanh u) / 2 is q where u is negative and 1 - q elsewhere, so that nothing cancels and
// nothing overflows. With the hardware's exponential and reciprocal the largest errors
// against 64 bits are 1.4e-7 over |x| < 4 and 2.4e-7 over |x| < 12 for gelu, 1.5e-7 for its
// slope; the general path's tanhf gives 2.9e-7, 4.3e-7 and 5.6e-7, and x / (1 + e^{-2u}) with
// its slope from 1 - s gave 4.2e-7, 5.2e-7 and 2.0e-6, in the same time.
struct GeluTail {
  float q, square;
};

__device__ inline GeluTail gelu_tail(float x) {
  constexpr float k = static_cast<float>(-2.0 / 0.6931471805599453 * 0.7978845608028654);
  const float square = x * x;
  const float cubic = x * __builtin_fmaf(kGeluA, square, 1.0f);
  const float e = __builtin_amdgcn_exp2f(k * __builtin_fabsf(cubic));
  return {e * __builtin_amdgcn_rcpf(1.0f + e), square};
}

// max(x, 0) - |x| q (the bound keeps an infinity, whose tail is zero, an infinity).
__device__ inline float gelu(float x, const GeluTail& t) {
  return __builtin_fmaf(-__builtin_fabsf(fminf(x, 3e38f)), t.q, fmaxf(x, 0.0f));
}

__device__ inline float gelu(float x) { return gelu(x, gelu_tail(x)); }

__device__ inline float gelu_slope(float x, const GeluTail& t) {
  constexpr float one = 2.0f * kGeluC, cube = 6.0f * kGeluC * kGeluA;
  const float rest = 1.0f - t.q;
  return __builtin_fmaf(x * t.q * rest, __builtin_fmaf(cube, t.square, one), x > 0.0f ? rest : t.q);
}

// The sum over the 16 lanes that share lane / 16.
__device__ inline float sum16(float v) {
  v += __shfl_xor(v, 1);
  v += __shfl_xor(v, 2);
  v += __shfl_xor(v, 4);
  v += __shfl_xor(v, 8);
  return v;
}

// A lane's eight spectral elements of one channel from the (MP, rows, WP) layout. (Eight
// together in a (rows, WP, MP) layout gain the layers nothing and cost the mixing's stores
// half its time again.)
__device__ inline v8b load_spectrum(const bf16* y, int k0, int b, int c, int rows, int WP) {
  us8 v;
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = y[(static_cast<long>(k0 + e) * rows + b) * WP + c];
  return __builtin_bit_cast(v8b, v);
}

// ------------------------------------------------------------------------ forward

struct LayerArgs {
  int W, H, n, NP, np, B, rows, per, chunks;
  const bf16* v_in;  // (B, NP, WP)
  const bf16* w;     // (WP, WP)
  const float* bias;
  const bf16* yhat;  // (MP, rows, WP)
  const bf16 *g_s, *f_k;
  bf16* v_out;       // null: not stored
  float* share;      // (chunks, MP, B, WP)
  // The lift.
  const float *spec, *prm, *pw, *pb;
  // The head.
  const bf16* q1;    // (kHeadUnits, WP)
  const float *b1, *q2, *q2b;
  float* out;
  const float* target;
  float *dout, *loss;
};

// One layer's forward pass over a run of tiles: v = act(W v_in + G yhat + bias), stored
// and contracted with the next layer's forward transform. LIFT forms the first
// activations from the inputs instead; HEAD (the last layer, linear) feeds the head, whose
// hidden units never leave the registers.
//
// Two workgroups a CU (launch bound) hide the tile's load latency behind the other's
// contraction; a wave takes half the channels and half the bins, so that each constant
// fragment (weights, spectra) is held by two waves and each streamed one loaded by two.
template <int WP, int MP, bool LIFT, bool HEAD>
__global__ void __launch_bounds__(256, 2) tile_layer(LayerArgs a) {
  constexpr int NC = WP / 32, KW = WP / 32, KM = MP / 32, MT = WP / 16, NT = MP / 64;
  constexpr int kCol = WP + 8;
  static_assert(wide_pitch<bf16>(kCol));
  __shared__ alignas(kWide) bf16 tile_cs[HEAD ? 1 : 2][HEAD ? 1 : WP * kRow];
  __shared__ alignas(kWide) bf16 tile_sc[HEAD ? 2 : 1][HEAD ? kTile * kCol : 1];
  __shared__ float red[4];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, q = lane >> 4, l16 = lane & 15;
  const int ws = wave >> 1, wc = wave & 1;
  const int b = blockIdx.x / a.chunks, chunk = blockIdx.x % a.chunks;
  const int first = chunk * a.per, last = min(first + a.per, a.NP / kTile);
  v8b wf[NC][KW], yf[NC][KM];
  float bias[NC][4], slope[NC][4], grid[NC][4];
#pragma unroll
  for (int j = 0; j < NC; ++j) {
    if constexpr (!LIFT) {
      const int c = wc * (WP / 2) + 16 * j + l16;
#pragma unroll
      for (int t = 0; t < KW; ++t) wf[j][t] = load8(a.w + c * WP + 32 * t + 8 * q);
#pragma unroll
      for (int t = 0; t < KM; ++t) yf[j][t] = load_spectrum(a.yhat, 32 * t + 8 * q, b, c, a.rows, WP);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int c = wc * (WP / 2) + 16 * j + 4 * q + r;
      const bool in = c < a.W;
      if (LIFT) {
        const float* row = a.pw + c * (a.np + 2);
        float fixed = in ? a.pb[c] : 0.f;
        for (int p = 0; in && p < a.np; ++p) fixed += row[1 + p] * a.prm[b * a.np + p];
        bias[j][r] = fixed;
        slope[j][r] = in ? row[0] : 0.f;
        grid[j][r] = in ? row[1 + a.np] : 0.f;
      } else {
        bias[j][r] = in ? a.bias[c] : 0.f;
      }
    }
  }
  v8b qf[HEAD ? 8 : 1][KW];
  float hb[HEAD ? 8 : 1], hq[HEAD ? 8 : 1], q2b = 0.f, loss = 0.f;
  if constexpr (HEAD) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int h = 16 * j + l16;
#pragma unroll
      for (int t = 0; t < KW; ++t) qf[j][t] = load8(a.q1 + h * WP + 32 * t + 8 * q);
      hb[j] = h < a.H ? a.b1[h] : 0.f;
      hq[j] = h < a.H ? a.q2[h] : 0.f;
    }
    q2b = a.q2b[0];
  }
  v4f sums[HEAD ? 1 : MT][HEAD ? 1 : NT] = {};
  const bf16* v_in = LIFT ? nullptr : a.v_in + static_cast<long>(b) * a.NP * WP;
  for (int tile = first; tile < last; ++tile) {
    const int buf = (tile - first) & 1;
    const int s0 = tile * kTile + ws * 32;
    v4f acc[NC][2] = {};
    if constexpr (!LIFT) {
      v8b gf[2][KM], vf[2][KW];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int s = s0 + 16 * i + l16;
#pragma unroll
        for (int t = 0; t < KW; ++t) vf[i][t] = load8(v_in + static_cast<long>(s) * WP + 32 * t + 8 * q);
#pragma unroll
        for (int t = 0; t < KM; ++t) gf[i][t] = load8(a.g_s + static_cast<long>(s) * MP + 32 * t + 8 * q);
      }
#pragma unroll
      for (int t = 0; t < KM; ++t)
#pragma unroll
        for (int j = 0; j < NC; ++j)
#pragma unroll
          for (int i = 0; i < 2; ++i) acc[j][i] = mfma(yf[j][t], gf[i][t], acc[j][i]);
#pragma unroll
      for (int t = 0; t < KW; ++t)
#pragma unroll
        for (int j = 0; j < NC; ++j)
#pragma unroll
          for (int i = 0; i < 2; ++i) acc[j][i] = mfma(wf[j][t], vf[i][t], acc[j][i]);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int s = s0 + 16 * i + l16, local = ws * 32 + 16 * i + l16;
      const bool in = s < a.n;
      float x = 0.f, at = 0.f;
      if (LIFT) {
        x = in ? a.spec[static_cast<long>(b) * a.n + s] : 0.f;
        at = static_cast<float>(s) / static_cast<float>(a.n);
      }
#pragma unroll
      for (int j = 0; j < NC; ++j) {
        const int c = wc * (WP / 2) + 16 * j + 4 * q;
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (LIFT)
            v[r] = slope[j][r] * x + bias[j][r] + grid[j][r] * at;
          else
            v[r] = acc[j][i][r] + bias[j][r];
          if (!LIFT && !HEAD) v[r] = gelu(v[r]);
          if (!in) v[r] = 0.f;  // bins beyond the grid hold nothing
        }
        const uint2 packed = bf4(v[0], v[1], v[2], v[3]);
        if (a.v_out)
          *reinterpret_cast<uint2*>(a.v_out + (static_cast<long>(b) * a.NP + s) * WP + c) = packed;
        if constexpr (HEAD) {
          *reinterpret_cast<uint2*>(&tile_sc[buf][local * kCol + c]) = packed;
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) tile_cs[buf][(c + r) * kRow + local] = bf(v[r]);
        }
      }
    }
    __syncthreads();  // the other buffer is free again: its readers are past this barrier
    if constexpr (HEAD) {
      v4f h[8] = {};
      const int row = 16 * wave;
#pragma unroll
      for (int t = 0; t < KW; ++t) {
        const v8b vf = load8(&tile_sc[buf][(row + l16) * kCol + 32 * t + 8 * q]);
#pragma unroll
        for (int j = 0; j < 8; ++j) h[j] = mfma(vf, qf[j][t], h[j]);
      }
      float o[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] += hq[j] * gelu(h[j][r] + hb[j]);
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = sum16(o[r]) + q2b;
      const float mine = l16 == 0 ? o[0] : l16 == 1 ? o[1] : l16 == 2 ? o[2] : o[3];
      const int s = tile * kTile + row + 4 * q + l16;
      if (l16 < 4 && s < a.n) {
        const long at = static_cast<long>(b) * a.n + s;
        a.out[at] = mine;
        if (a.target) {
          const float d = mine - a.target[at];
          a.dout[at] = 2.0f * d / static_cast<float>(static_cast<long>(a.B) * a.n);
          loss += d * d;
        }
      }
    } else {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        v8b ff[NT];
#pragma unroll
        for (int k = 0; k < NT; ++k)
          ff[k] = load8(a.f_k + static_cast<long>(16 * (wave * NT + k) + l16) * a.NP +
                        tile * kTile + 32 * t + 8 * q);
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          const v8b vf = load8(&tile_cs[buf][(16 * m + l16) * kRow + 32 * t + 8 * q]);
#pragma unroll
          for (int k = 0; k < NT; ++k) sums[m][k] = mfma(vf, ff[k], sums[m][k]);
        }
      }
    }
  }
  if constexpr (HEAD) {
    if (a.target) {
      loss = sum16(loss);
      loss += __shfl_xor(loss, 16);
      loss += __shfl_xor(loss, 32);
      if (lane == 0) red[wave] = loss;
      __syncthreads();
      if (tid == 0) a.loss[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
    }
  } else {
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int k = 0; k < NT; ++k) {
        const long k2 = 16 * (wave * NT + k) + l16;
        *reinterpret_cast<v4f*>(a.share + ((chunk * static_cast<long>(MP) + k2) * a.B + b) * WP +
                                16 * m + 4 * q) = sums[m][k];
      }
  }
}

__global__ void tile_loss(const float* __restrict__ partials, int n, long count,
                          float* __restrict__ loss) {
  __shared__ float red[256];
  float e = 0.f;
  for (int i = threadIdx.x; i < n; i += blockDim.x) e += partials[i];
  red[threadIdx.x] = e;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) *loss = red[0] / static_cast<float>(count);
}

// ------------------------------------------------------------------------- mixing

struct MixArgs {
  int W, M, B, rows, chunks;
  const float* share;  // (chunks, MP, B, WP)
  float* total;        // the shares' sum (MP, B, WP); null: not kept
  const float *rre, *rim;
  bf16* mixed;         // (MP, rows, WP)
};

// One mode and 16 samples a workgroup: the workgroups' spectral shares summed in order,
// then the complex product with the mode's weights on the FP32 matrix cores
// (v_mfma_f32_16x16x4_f32; a wave takes 16 output channels). BACK multiplies by the
// conjugate transpose. The weights are read once per 16 samples, each in 64-byte runs.
template <int WP, int MP, bool BACK>
__global__ void __launch_bounds__(256) tile_mix(MixArgs a) {
  constexpr int kCol = WP + 4;
  __shared__ alignas(kWide) float in[2][16 * kCol];
  static_assert(wide_pitch<float>(kCol));
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, q = lane >> 4, l16 = lane & 15;
  const int k = blockIdx.x, b0 = blockIdx.y * 16;
  const long plane = static_cast<long>(MP) * a.B * WP;
  // The wave's weights first, all at once: they wait for nothing, and the shares' loads
  // (eight in flight, added in order) overlap theirs. Loaded between the products they were
  // most of the kernel's 12.1 us at 64 channels and samples; now 6.5 us.
  const int o = 16 * wave + l16;
  float wr[WP / 4], wi[WP / 4];
  if (wave < WP / 16) {
#pragma unroll
    for (int n = 0; n < WP / 4; ++n) {
      const int i = 16 * (n / 4) + 4 * q + n % 4;
      const bool have = i < a.W && o < a.W;
      const long at = BACK ? (static_cast<long>(k) * a.W + o) * a.W + i
                           : (static_cast<long>(k) * a.W + i) * a.W + o;
      wr[n] = have ? a.rre[at] : 0.f;
      wi[n] = have ? a.rim[at] : 0.f;
    }
  }
  for (int e = tid; e < 2 * 16 * WP / 4; e += 256) {
    const int part = e / (16 * WP / 4), row = e / (WP / 4) % 16, c = e % (WP / 4) * 4;
    v4f v = {0.f, 0.f, 0.f, 0.f};
    if (b0 + row < a.B) {
      const long at = (static_cast<long>(k + part * (MP / 2)) * a.B + b0 + row) * WP + c;
#pragma unroll 8
      for (int z = 0; z < a.chunks; ++z)
        v += *reinterpret_cast<const v4f*>(a.share + z * plane + at);
      if (a.total) *reinterpret_cast<v4f*>(a.total + at) = v;
    }
    *reinterpret_cast<v4f*>(&in[part][row * kCol + c]) = v;
  }
  __syncthreads();
  if (wave >= WP / 16) return;
  v4f yr = {0.f, 0.f, 0.f, 0.f}, yi = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < WP / 16; ++t) {
    const v4f vr = *reinterpret_cast<const v4f*>(&in[0][l16 * kCol + 16 * t + 4 * q]);
    const v4f vi = *reinterpret_cast<const v4f*>(&in[1][l16 * kCol + 16 * t + 4 * q]);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float rr = wr[4 * t + r], ri = wi[4 * t + r];
      yr = mfma32(vr[r], rr, yr);
      yi = mfma32(vi[r], rr, yi);
      yr = mfma32(BACK ? vi[r] : -vi[r], ri, yr);
      yi = mfma32(BACK ? -vr[r] : vr[r], ri, yi);
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int b = b0 + 4 * q + r;
    if (b >= a.B) continue;
    a.mixed[(static_cast<long>(k) * a.rows + b) * WP + o] = bf(yr[r]);
    a.mixed[(static_cast<long>(MP / 2 + k) * a.rows + b) * WP + o] = bf(yi[r]);
  }
}

// The spectral weights' gradient, conj(vhat)^T dyhat over the batch: one mode, 16 input
// channels and a layer a workgroup, a wave 16 output channels.
template <int WP, int MP>
__global__ void __launch_bounds__(256) tile_mix_weight(const float* __restrict__ vhat,
                                                       const float* __restrict__ dyhat,
                                                       long layer_stride, float* __restrict__ gre,
                                                       float* __restrict__ gim, long grad_stride,
                                                       int W, int B) {
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, q = lane >> 4, l16 = lane & 15;
  if (wave >= WP / 16) return;
  const int k = blockIdx.x, i0 = blockIdx.y * 16, layer = blockIdx.z;
  const float* vr = vhat + layer * layer_stride + static_cast<long>(k) * B * WP + i0 + l16;
  const float* yr = dyhat + layer * layer_stride + static_cast<long>(k) * B * WP + 16 * wave + l16;
  const long imag = static_cast<long>(MP / 2) * B * WP;
  v4f re = {0.f, 0.f, 0.f, 0.f}, im = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
  for (int b0 = 0; b0 < B; b0 += 4) {
    const int b = b0 + q;
    const bool in = b < B;
    const long at = static_cast<long>(b) * WP;
    const float ar = in ? vr[at] : 0.f, ai = in ? vr[imag + at] : 0.f;
    const float br = in ? yr[at] : 0.f, bi = in ? yr[imag + at] : 0.f;
    re = mfma32(ar, br, re);
    im = mfma32(ar, bi, im);
    re = mfma32(ai, bi, re);
    im = mfma32(-ai, br, im);
  }
  const int o = 16 * wave + l16;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int i = i0 + 4 * q + r;
    if (i >= W || o >= W) continue;
    const long at = layer * grad_stride + (static_cast<long>(k) * W + i) * W + o;
    gre[at] = re[r];
    gim[at] = im[r];
  }
}

// ----------------------------------------------------------------------- backward

struct HeadBackArgs {
  int H, n, NP, per, chunks;
  const bf16* v;     // (B, NP, WP), the head's input
  const float* dout;
  const bf16 *q1, *q1t;
  const float *b1, *q2;
  bf16* dz;          // (B, NP, WP)
  float* dq;         // per workgroup: (kHeadUnits, WP), kHeadUnits, kHeadUnits, WP, 1
};

// The head's backward pass over a run of tiles: the hidden units recomputed, their
// gradient handed over in LDS both ways round, dv = Q1^T dh (the last layer is linear, so
// this is its dz), and the weights' sums in registers over the run.
template <int WP>
__global__ void __launch_bounds__(256, 1) tile_head_backward(HeadBackArgs a) {
  constexpr int NC = WP / 32, KW = WP / 32, MT = WP / 16;
  constexpr int kHid = kHeadUnits + 8;
  static_assert(wide_pitch<bf16>(kHid));
  __shared__ alignas(kWide) bf16 dh_hs[2][kHeadUnits * kRow];
  __shared__ alignas(kWide) bf16 dh_sh[2][kTile * kHid];
  __shared__ alignas(kWide) bf16 v_cs[2][WP * kRow];
  __shared__ float red[2 * kHeadUnits + WP + 1];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, q = lane >> 4, l16 = lane & 15;
  const int ws = wave >> 1, wc = wave & 1;
  const int b = blockIdx.x / a.chunks, chunk = blockIdx.x % a.chunks;
  const int first = chunk * a.per, last = min(first + a.per, a.NP / kTile);
  v8b qf[4][KW], qtf[NC][4];
  float hb[4], hq[4], db[4] = {}, dq2[4] = {}, dbl[NC][4] = {}, dsum = 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int h = wc * 64 + 16 * j + l16;
#pragma unroll
    for (int t = 0; t < KW; ++t) qf[j][t] = load8(a.q1 + h * WP + 32 * t + 8 * q);
    hb[j] = h < a.H ? a.b1[h] : 0.f;
    hq[j] = h < a.H ? a.q2[h] : 0.f;
  }
#pragma unroll
  for (int j = 0; j < NC; ++j)
#pragma unroll
    for (int t = 0; t < 4; ++t)
      qtf[j][t] = load8(a.q1t + (wc * (WP / 2) + 16 * j + l16) * kHeadUnits + 32 * t + 8 * q);
  v4f dq[2][MT] = {};
  const bf16* v = a.v + static_cast<long>(b) * a.NP * WP;
  for (int tile = first; tile < last; ++tile) {
    const int buf = (tile - first) & 1;
    const int s0 = tile * kTile + ws * 32;
    v8b vf[2][KW];
    float d[2][4];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
      for (int t = 0; t < KW; ++t)
        vf[i][t] = load8(v + static_cast<long>(s0 + 16 * i + l16) * WP + 32 * t + 8 * q);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int s = s0 + 16 * i + 4 * q + r;
        d[i][r] = s < a.n ? a.dout[static_cast<long>(b) * a.n + s] : 0.f;
        dsum += d[i][r];
      }
    }
    // The bins' rows turned for the contraction over bins, half of the channels a wave.
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int t = 0; t < KW; ++t)
        if (t == wc || (KW == 1 && wc == 0)) {
          const us8 u = __builtin_bit_cast(us8, vf[i][t]);
#pragma unroll
          for (int e = 0; e < 8; ++e)
            v_cs[buf][(32 * t + 8 * q + e) * kRow + ws * 32 + 16 * i + l16] = u[e];
        }
    v4f h[2][4] = {};
#pragma unroll
    for (int t = 0; t < KW; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 2; ++i) h[i][j] = mfma(vf[i][t], qf[j][t], h[i][j]);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int hu = wc * 64 + 16 * j + l16, local = ws * 32 + 16 * i + 4 * q;
        float g[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float x = h[i][j][r] + hb[j];
          const GeluTail tail = gelu_tail(x);
          g[r] = hq[j] * d[i][r] * gelu_slope(x, tail);
          db[j] += g[r];
          dq2[j] += d[i][r] * gelu(x, tail);
          dh_sh[buf][(local + r) * kHid + hu] = bf(g[r]);
        }
        *reinterpret_cast<uint2*>(&dh_hs[buf][hu * kRow + local]) = bf4(g[0], g[1], g[2], g[3]);
      }
    __syncthreads();
    v4f dv[NC][2] = {};
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const v8b hf = load8(&dh_sh[buf][(ws * 32 + 16 * i + l16) * kHid + 32 * t + 8 * q]);
#pragma unroll
        for (int j = 0; j < NC; ++j) dv[j][i] = mfma(qtf[j][t], hf, dv[j][i]);
      }
#pragma unroll
    for (int j = 0; j < NC; ++j)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int s = s0 + 16 * i + l16, c = wc * (WP / 2) + 16 * j + 4 * q;
#pragma unroll
        for (int r = 0; r < 4; ++r) dbl[j][r] += dv[j][i][r];
        *reinterpret_cast<uint2*>(a.dz + (static_cast<long>(b) * a.NP + s) * WP + c) =
            bf4(dv[j][i][0], dv[j][i][1], dv[j][i][2], dv[j][i][3]);
      }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      v8b hf[2];
#pragma unroll
      for (int m = 0; m < 2; ++m)
        hf[m] = load8(&dh_hs[buf][(32 * wave + 16 * m + l16) * kRow + 32 * t + 8 * q]);
#pragma unroll
      for (int k = 0; k < MT; ++k) {
        const v8b cf = load8(&v_cs[buf][(16 * k + l16) * kRow + 32 * t + 8 * q]);
#pragma unroll
        for (int m = 0; m < 2; ++m) dq[m][k] = mfma(hf[m], cf, dq[m][k]);
      }
    }
  }
  float* share = a.dq + blockIdx.x * head_share(WP);
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int k = 0; k < MT; ++k)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        share[(32 * wave + 16 * m + 4 * q + r) * WP + 16 * k + l16] = dq[m][k][r];
  // The vector sums: over the lanes, then the first half's bins plus the second's.
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    db[j] += __shfl_xor(db[j], 16);
    db[j] += __shfl_xor(db[j], 32);
    dq2[j] += __shfl_xor(dq2[j], 16);
    dq2[j] += __shfl_xor(dq2[j], 32);
  }
  dsum += __shfl_xor(dsum, 16);
  dsum += __shfl_xor(dsum, 32);
#pragma unroll
  for (int j = 0; j < NC; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) dbl[j][r] = sum16(dbl[j][r]);
  for (int half = 0; half < 2; ++half) {
    __syncthreads();
    if (ws != half) continue;
    auto put = [&](int at, float x) { red[at] = half ? red[at] + x : x; };
    if (q == 0)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        put(wc * 64 + 16 * j + l16, db[j]);
        put(kHeadUnits + wc * 64 + 16 * j + l16, dq2[j]);
      }
    if (l16 == 0)
#pragma unroll
      for (int j = 0; j < NC; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          put(2 * kHeadUnits + wc * (WP / 2) + 16 * j + 4 * q + r, dbl[j][r]);
    if (wc == 0 && lane == 0) put(2 * kHeadUnits + WP, dsum);
  }
  __syncthreads();
  for (int e = tid; e < 2 * kHeadUnits + WP + 1; e += 256) share[kHeadUnits * WP + e] = red[e];
}

struct BackArgs {
  int W, n, NP, np, B, rows, per, chunks;
  // The layer above: its dz, its convolution's transpose and its spectral gradient.
  const bf16 *dz_in, *wt, *dvhat, *f_s;
  // This layer: input, convolution, bias and mixed spectrum (the pre-activation's parts).
  const bf16 *v, *w, *yhat, *g_s;
  const float* bias;
  bf16* dz;          // this layer's dz, (B, NP, WP)
  const bf16* g_k;
  float* share;      // (chunks, MP, B, WP)
  float* dw;         // per workgroup: (WP, WP), then WP
  // The lift.
  const float* spec;
  float* dlift;      // per workgroup: (3, WP)
};

enum class Back { kTop, kLayer, kLift };

// One layer's backward pass over a run of tiles. kLayer forms
// dz = (W'^T dz' + F dvhat') gelu'(z), z recomputed, and stores it; kTop takes the dz the
// head's pass stored. Both contract dz with the layer's input (the convolution's
// gradient) and with the inverse transform (its spectrum's), in registers over the run.
// kLift ends the chain with the lift's sums.
// kLayer keeps up to 300 registers a lane of constants and sums: one workgroup a CU.
template <int WP, int MP, Back MODE>
__global__ void __launch_bounds__(256, MODE == Back::kLayer ? 1 : 2)
    tile_backward_layer(BackArgs a) {
  constexpr int NC = WP / 32, KW = WP / 32, KM = MP / 32, MT = WP / 16, NT = MP / 64;
  constexpr int kOwn = MT * MT / 4;  // tiles of the convolution's gradient a wave sums
  constexpr bool kTop = MODE == Back::kTop, kLift = MODE == Back::kLift;
  __shared__ alignas(kWide) bf16 dz_cs[2][kLift ? 1 : WP * kRow];
  __shared__ alignas(kWide) bf16 v_cs[2][kLift ? 1 : WP * kRow];
  __shared__ float red[3 * WP];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, q = lane >> 4, l16 = lane & 15;
  const int ws = wave >> 1, wc = wave & 1;
  const int b = blockIdx.x / a.chunks, chunk = blockIdx.x % a.chunks;
  const int first = chunk * a.per, last = min(first + a.per, a.NP / kTile);
  v8b wtf[NC][KW], dvf[NC][KM], wf[NC][KW], yf[NC][KM];
  float bias[NC][4], db[NC][4] = {}, dspec[NC][4] = {}, dgrid[NC][4] = {};
  if constexpr (!kTop) {
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      const int c = wc * (WP / 2) + 16 * j + l16;
#pragma unroll
      for (int t = 0; t < KW; ++t) wtf[j][t] = load8(a.wt + c * WP + 32 * t + 8 * q);
#pragma unroll
      for (int t = 0; t < KM; ++t) dvf[j][t] = load_spectrum(a.dvhat, 32 * t + 8 * q, b, c, a.rows, WP);
      if constexpr (!kLift) {
#pragma unroll
        for (int t = 0; t < KW; ++t) wf[j][t] = load8(a.w + c * WP + 32 * t + 8 * q);
#pragma unroll
        for (int t = 0; t < KM; ++t)
          yf[j][t] = load_spectrum(a.yhat, 32 * t + 8 * q, b, c, a.rows, WP);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = wc * (WP / 2) + 16 * j + 4 * q + r;
          bias[j][r] = row < a.W ? a.bias[row] : 0.f;
        }
      }
    }
  }
  v4f dw[kLift ? 1 : kOwn] = {}, sums[kLift ? 1 : MT][kLift ? 1 : NT] = {};
  const long base = static_cast<long>(b) * a.NP * WP;
  for (int tile = first; tile < last; ++tile) {
    const int buf = (tile - first) & 1;
    const int s0 = tile * kTile + ws * 32;
    v8b zf[2][KW], vf[2][KW];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int t = 0; t < KW; ++t) {
        const long at = base + static_cast<long>(s0 + 16 * i + l16) * WP + 32 * t + 8 * q;
        zf[i][t] = load8(a.dz_in + at);
        if (!kLift) vf[i][t] = load8(a.v + at);
      }
    v4f dv[NC][2] = {}, z[NC][2] = {};
    if constexpr (!kTop) {
#pragma unroll
      for (int t = 0; t < KM; ++t)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const long at = static_cast<long>(s0 + 16 * i + l16) * MP + 32 * t + 8 * q;
          const v8b ff = load8(a.f_s + at);
#pragma unroll
          for (int j = 0; j < NC; ++j) dv[j][i] = mfma(dvf[j][t], ff, dv[j][i]);
          if constexpr (!kLift) {
            const v8b gf = load8(a.g_s + at);
#pragma unroll
            for (int j = 0; j < NC; ++j) z[j][i] = mfma(yf[j][t], gf, z[j][i]);
          }
        }
#pragma unroll
      for (int t = 0; t < KW; ++t)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < NC; ++j) {
            dv[j][i] = mfma(wtf[j][t], zf[i][t], dv[j][i]);
            if (!kLift) z[j][i] = mfma(wf[j][t], vf[i][t], z[j][i]);
          }
    }
    if constexpr (kLift) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int s = s0 + 16 * i + l16;
        const float x = s < a.n ? a.spec[static_cast<long>(b) * a.n + s] : 0.f;
        const float at = static_cast<float>(s) / static_cast<float>(a.n);
#pragma unroll
        for (int j = 0; j < NC; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            dspec[j][r] += dv[j][i][r] * x;
            dgrid[j][r] += dv[j][i][r] * at;
            db[j][r] += dv[j][i][r];
          }
      }
      continue;
    }
    // The input's rows turned for the contraction over bins, half of the channels a wave
    // (and the top layer's dz with them).
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int t = 0; t < KW; ++t)
        if (t == wc || (KW == 1 && wc == 0)) {
          const us8 u = __builtin_bit_cast(us8, vf[i][t]);
          const us8 d = __builtin_bit_cast(us8, zf[i][t]);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const int at = (32 * t + 8 * q + e) * kRow + ws * 32 + 16 * i + l16;
            v_cs[buf][at] = u[e];
            if (kTop) dz_cs[buf][at] = d[e];
          }
        }
    if constexpr (!kTop) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int s = s0 + 16 * i + l16, local = ws * 32 + 16 * i + l16;
#pragma unroll
        for (int j = 0; j < NC; ++j) {
          const int c = wc * (WP / 2) + 16 * j + 4 * q;
          float d[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float x = z[j][i][r] + bias[j][r];
            d[r] = dv[j][i][r] * gelu_slope(x, gelu_tail(x));
            if (s >= a.n) d[r] = 0.f;
            db[j][r] += d[r];
            dz_cs[buf][(c + r) * kRow + local] = bf(d[r]);
          }
          *reinterpret_cast<uint2*>(a.dz + base + static_cast<long>(s) * WP + c) =
              bf4(d[0], d[1], d[2], d[3]);
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      v8b gf[NT];
#pragma unroll
      for (int k = 0; k < NT; ++k)
        gf[k] = load8(a.g_k + static_cast<long>(16 * (wave * NT + k) + l16) * a.NP + tile * kTile +
                      32 * t + 8 * q);
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const v8b df = load8(&dz_cs[buf][(16 * m + l16) * kRow + 32 * t + 8 * q]);
#pragma unroll
        for (int k = 0; k < NT; ++k) sums[m][k] = mfma(df, gf[k], sums[m][k]);
      }
#pragma unroll
      for (int o = 0; o < kOwn; ++o) {
        const int m = (wave + 4 * o) / MT, k = (wave + 4 * o) % MT;
        const v8b df = load8(&dz_cs[buf][(16 * m + l16) * kRow + 32 * t + 8 * q]);
        const v8b cf = load8(&v_cs[buf][(16 * k + l16) * kRow + 32 * t + 8 * q]);
        dw[o] = mfma(df, cf, dw[o]);
      }
    }
  }
  if constexpr (!kLift) {
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int k = 0; k < NT; ++k) {
        const long k2 = 16 * (wave * NT + k) + l16;
        *reinterpret_cast<v4f*>(a.share + ((chunk * static_cast<long>(MP) + k2) * a.B + b) * WP +
                                16 * m + 4 * q) = sums[m][k];
      }
    float* own = a.dw + static_cast<long>(blockIdx.x) * (WP * WP + WP);
#pragma unroll
    for (int o = 0; o < kOwn; ++o) {
      const int m = (wave + 4 * o) / MT, k = (wave + 4 * o) % MT;
#pragma unroll
      for (int r = 0; r < 4; ++r) own[(16 * m + 4 * q + r) * WP + 16 * k + l16] = dw[o][r];
    }
  }
  if (kTop) return;  // the head's pass summed this layer's bias
  // The bias sums (and the lift's): over the lanes, then the first half's bins plus the
  // second's.
#pragma unroll
  for (int j = 0; j < NC; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      db[j][r] = sum16(db[j][r]);
      if constexpr (kLift) {
        dspec[j][r] = sum16(dspec[j][r]);
        dgrid[j][r] = sum16(dgrid[j][r]);
      }
    }
  for (int half = 0; half < 2; ++half) {
    __syncthreads();
    if (ws != half || l16 != 0) continue;
#pragma unroll
    for (int j = 0; j < NC; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int c = wc * (WP / 2) + 16 * j + 4 * q + r;
        red[c] = half ? red[c] + db[j][r] : db[j][r];
        if constexpr (kLift) {
          red[WP + c] = half ? red[WP + c] + dspec[j][r] : dspec[j][r];
          red[2 * WP + c] = half ? red[2 * WP + c] + dgrid[j][r] : dgrid[j][r];
        }
      }
  }
  __syncthreads();
  float* to = kLift ? a.dlift + static_cast<long>(blockIdx.x) * 3 * WP
                    : a.dw + static_cast<long>(blockIdx.x) * (WP * WP + WP) + WP * WP;
  for (int e = tid; e < (kLift ? 3 : 1) * WP; e += 256) to[e] = red[e];
}

// The workgroups' weight-gradient shares summed in workgroup order, 64 outputs a block:
// four runs of workgroups side by side, then the runs in order.
__global__ void __launch_bounds__(256) tile_gradient(const GradientSegment* __restrict__ segments,
                                                     int count, int groups, int chunks,
                                                     const float* __restrict__ prm, int np) {
  __shared__ float red[4][64];
  int at = 0;
  while (at + 1 < count && static_cast<int>(blockIdx.x) >= segments[at + 1].first_block) ++at;
  const GradientSegment g = segments[at];
  const int e = (blockIdx.x - g.first_block) * 64 + (threadIdx.x & 63), run = threadIdx.x >> 6;
  const bool in = e < g.rows * g.cols;
  const int row = in ? e / g.cols : 0, col = in ? e % g.cols : 0;
  const float* src = g.src + static_cast<long>(row) * g.src_ld + col;
  const int per = (groups + 3) / 4, from = run * per, to = min(groups, from + per);
  float v = 0.f;
  if (in) {
    if (g.scan_parameter < 0) {
#pragma unroll 16
      for (int w = from; w < to; ++w) v += src[w * g.stride];
    } else {
      for (int w = from; w < to; ++w)
        v += prm[(w / chunks) * np + g.scan_parameter] * src[w * g.stride];
    }
  }
  red[run][threadIdx.x & 63] = v;
  __syncthreads();
  if (run == 0 && in) {
    const int l = threadIdx.x;
    g.dst[static_cast<long>(row) * g.dst_ld + col] = ((red[0][l] + red[1][l]) + red[2][l]) + red[3][l];
  }
}

// The padded BF16 copies of the convolutions (blocks below `layers`) and the head.
struct PackArgs {
  const float* param;
  long w0, w_stride, q1;
  bf16 *w, *wt, *q1p, *q1t;
  int W, H, WP, layers;
};

__global__ void tile_pack_kernel(PackArgs a) {
  const int layer = blockIdx.y;
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (layer < a.layers) {
    if (e >= a.WP * a.WP) return;
    const int o = e / a.WP, i = e % a.WP;
    const bf16 v = bf(o < a.W && i < a.W ? a.param[a.w0 + layer * a.w_stride + o * a.W + i] : 0.f);
    a.w[static_cast<long>(layer) * a.WP * a.WP + e] = v;
    a.wt[static_cast<long>(layer) * a.WP * a.WP + i * a.WP + o] = v;
  } else {
    if (e >= kHeadUnits * a.WP) return;
    const int h = e / a.WP, c = e % a.WP;
    const bf16 v = bf(h < a.H && c < a.W ? a.param[a.q1 + h * a.W + c] : 0.f);
    a.q1p[e] = v;
    a.q1t[c * kHeadUnits + h] = v;
  }
}

template <int WP, int MP>
void forward_impl(const TileShape& t, const Offsets& off, const float* param,
                  const TileBuffers& b, const float* spec, const float* prm, float* out,
                  const float* target, float* dout, float* loss, int B, bool keep,
                  hipStream_t stream) {
  const int layers = static_cast<int>(b.w.size());
  const TileSplit split = tile_split(t, B, kForwardGroups);
  const dim3 grid(static_cast<unsigned>(B * split.chunks));
  LayerArgs a{};
  a.W = t.W; a.H = t.H; a.n = t.n; a.NP = t.NP; a.np = t.np; a.B = B; a.rows = b.rows;
  a.per = split.per; a.chunks = split.chunks;
  a.g_s = b.g_s; a.f_k = b.f_k; a.share = b.share;
  a.spec = spec; a.prm = prm; a.pw = param + off.lift_w; a.pb = param + off.lift_b;
  a.v_out = b.v[0];
  hipLaunchKernelGGL(HIP_KERNEL_NAME(tile_layer<WP, MP, true, false>), grid, dim3(256), 0, stream, a);
  SP_HIP(hipGetLastError());
  for (int l = 0; l < layers; ++l) {
    const MixArgs m{t.W, t.M, B, b.rows, split.chunks, b.share, keep ? b.vhat[l] : nullptr,
                    param + off.r_re[l], param + off.r_im[l], b.yhat[l]};
    hipLaunchKernelGGL(HIP_KERNEL_NAME(tile_mix<WP, MP, false>), dim3(t.M, (B + 15) / 16), dim3(256),
                       0, stream, m);
    SP_HIP(hipGetLastError());
    a.v_in = b.v[l];
    a.w = b.w[l];
    a.bias = param + off.b[l];
    a.yhat = b.yhat[l];
    if (l + 1 < layers) {
      a.v_out = b.v[l + 1];
      hipLaunchKernelGGL(HIP_KERNEL_NAME(tile_layer<WP, MP, false, false>), grid, dim3(256), 0, stream,
                         a);
    } else {
      a.v_out = keep ? b.v[l + 1] : nullptr;
      a.q1 = b.q1; a.b1 = param + off.q1_b; a.q2 = param + off.q2_w; a.q2b = param + off.q2_b;
      a.out = out; a.target = target; a.dout = dout; a.loss = b.loss;
      hipLaunchKernelGGL(HIP_KERNEL_NAME(tile_layer<WP, MP, false, true>), grid, dim3(256), 0, stream,
                         a);
    }
    SP_HIP(hipGetLastError());
  }
  if (target) {
    hipLaunchKernelGGL(tile_loss, dim3(1), dim3(256), 0, stream, b.loss,
                       static_cast<int>(grid.x), static_cast<long>(B) * t.n, loss);
    SP_HIP(hipGetLastError());
  }
}

template <int WP, int MP>
void backward_impl(const TileShape& t, const Offsets& off, const float* param, float* grad,
                   const TileBuffers& b, const float* spec, const float* prm, const float* dout,
                   int B, hipStream_t stream) {
  const int layers = static_cast<int>(b.w.size());
  const TileSplit split = tile_split(t, B, kBackwardGroups);
  const dim3 grid(static_cast<unsigned>(B * split.chunks));
  const HeadBackArgs h{t.H, t.n, t.NP, split.per, split.chunks, b.v[layers], dout, b.q1, b.q1t,
                       param + off.q1_b, param + off.q2_w, b.dz[0], b.dq};
  hipLaunchKernelGGL(HIP_KERNEL_NAME(tile_head_backward<WP>), grid, dim3(256), 0, stream, h);
  SP_HIP(hipGetLastError());
  BackArgs a{};
  a.W = t.W; a.n = t.n; a.NP = t.NP; a.np = t.np; a.B = B; a.rows = b.rows;
  a.per = split.per; a.chunks = split.chunks;
  a.f_s = b.f_s; a.g_s = b.g_s; a.g_k = b.g_k; a.share = b.share; a.dvhat = b.dvhat;
  a.spec = spec; a.dlift = b.dlift;
  int held = 0;  // the buffer the layer above left its dz in
  for (int l = layers - 1; l >= 0; --l) {
    a.v = b.v[l];
    a.w = b.w[l];
    a.yhat = b.yhat[l];
    a.bias = param + off.b[l];
    a.dw = b.dw[l];
    a.dz_in = b.dz[held];
    if (l == layers - 1) {
      hipLaunchKernelGGL(HIP_KERNEL_NAME(tile_backward_layer<WP, MP, Back::kTop>), grid, dim3(256), 0,
                         stream, a);
    } else {
      a.wt = b.wt[l + 1];
      a.dz = b.dz[held ^ 1];
      hipLaunchKernelGGL(HIP_KERNEL_NAME(tile_backward_layer<WP, MP, Back::kLayer>), grid, dim3(256),
                         0, stream, a);
      held ^= 1;
    }
    SP_HIP(hipGetLastError());
    const MixArgs m{t.W, t.M, B, b.rows, split.chunks, b.share, b.dyhat[l], param + off.r_re[l],
                    param + off.r_im[l], b.dvhat};
    hipLaunchKernelGGL(HIP_KERNEL_NAME(tile_mix<WP, MP, true>), dim3(t.M, (B + 15) / 16), dim3(256), 0,
                       stream, m);
    SP_HIP(hipGetLastError());
  }
  a.dz_in = b.dz[held];
  a.wt = b.wt[0];
  hipLaunchKernelGGL(HIP_KERNEL_NAME(tile_backward_layer<WP, MP, Back::kLift>), grid, dim3(256), 0,
                     stream, a);
  SP_HIP(hipGetLastError());
  const long layer_stride = layers > 1 ? b.vhat[1] - b.vhat[0] : 0;
  const long grad_stride = layers > 1 ? off.r_re[1] - off.r_re[0] : 0;
  hipLaunchKernelGGL(HIP_KERNEL_NAME(tile_mix_weight<WP, MP>), dim3(t.M, WP / 16, layers), dim3(256), 0,
                     stream, b.vhat[0], b.dyhat[0], layer_stride, grad + off.r_re[0],
                     grad + off.r_im[0], grad_stride, t.W, B);
  SP_HIP(hipGetLastError());
  hipLaunchKernelGGL(tile_gradient, dim3(b.segment_blocks), dim3(256), 0, stream, b.segments,
                     b.n_segments, static_cast<int>(grid.x), split.chunks, prm, t.np);
  SP_HIP(hipGetLastError());
}

template <typename F>
void dispatch(const TileShape& t, F&& f) {
  if (t.WP == 32 && t.MP == 64)
    f.template operator()<32, 64>();
  else if (t.WP == 32)
    f.template operator()<32, 128>();
  else if (t.MP == 64)
    f.template operator()<64, 64>();
  else
    f.template operator()<64, 128>();
}

struct ForwardCall {
  const TileShape& t; const Offsets& off; const float* param; const TileBuffers& b;
  const float *spec, *prm; float* out; const float* target; float *dout, *loss; int B; bool keep;
  hipStream_t stream;
  template <int WP, int MP>
  void operator()() const {
    forward_impl<WP, MP>(t, off, param, b, spec, prm, out, target, dout, loss, B, keep, stream);
  }
};

struct BackwardCall {
  const TileShape& t; const Offsets& off; const float* param; float* grad; const TileBuffers& b;
  const float *spec, *prm, *dout; int B; hipStream_t stream;
  template <int WP, int MP>
  void operator()() const {
    backward_impl<WP, MP>(t, off, param, grad, b, spec, prm, dout, B, stream);
  }
};

}  // namespace

// The tiles hold a layer's channels and modes whole: 64 channels by 128 spectral sums are
// what two workgroups a CU keep in registers. Wider networks take the general products: a
// training step of 64 samples of 2048 bins takes 0.52 ms at 64 channels, 64 modes and 128
// units, and 4.4 to 4.9 ms with one channel, mode or unit more. Within, padding costs
// little: 0.26 ms at 16 channels, 8 modes and 32 units (2.3 by the general products).
bool tile_available(const Shape& s) {
  return s.width <= 64 && s.modes <= 64 && s.hidden <= kHeadUnits;
}

TileShape tile_shape(const Shape& s) {
  TileShape t{};
  t.W = s.width; t.M = s.modes; t.H = s.hidden; t.n = s.n; t.np = s.n_params;
  t.WP = s.width <= 32 ? 32 : 64;
  t.MP = s.modes <= 32 ? 64 : 128;
  t.NP = (s.n + kTile - 1) / kTile * kTile;
  return t;
}

TileSplit tile_split(const TileShape& t, int batch, int workgroups) {
  const int tiles = t.NP / kTile;
  const int want = std::max(1, std::min(tiles, workgroups / batch));
  TileSplit s{};
  s.per = (tiles + want - 1) / want;
  s.chunks = (tiles + s.per - 1) / s.per;
  return s;
}

long tile_groups(int max_batch) {
  // chunks <= workgroups / batch (or one), so a batch takes at most max(workgroups, batch).
  return std::max({kForwardGroups, kBackwardGroups, max_batch});
}

void tile_pack(const TileShape& t, const Offsets& off, const float* param, const TileBuffers& b,
               hipStream_t stream) {
  PackArgs a{};
  a.param = param;
  a.w0 = off.w[0];
  a.w_stride = off.w.size() > 1 ? off.w[1] - off.w[0] : 0;
  a.q1 = off.q1_w;
  a.w = b.w[0]; a.wt = b.wt[0]; a.q1p = b.q1; a.q1t = b.q1t;
  a.W = t.W; a.H = t.H; a.WP = t.WP;
  a.layers = static_cast<int>(b.w.size());
  hipLaunchKernelGGL(tile_pack_kernel, dim3((kHeadUnits * t.WP + 255) / 256, a.layers + 1),
                     dim3(256), 0, stream, a);
  SP_HIP(hipGetLastError());
}

void tile_forward(const TileShape& t, const Offsets& off, const float* param,
                  const TileBuffers& b, const float* spec, const float* prm, float* out,
                  const float* target, float* dout, float* loss, int batch, bool keep,
                  hipStream_t stream) {
  dispatch(t, ForwardCall{t, off, param, b, spec, prm, out, target, dout, loss, batch, keep, stream});
}

void tile_backward(const TileShape& t, const Offsets& off, const float* param, float* grad,
                   const TileBuffers& b, const float* spec, const float* prm, const float* dout,
                   int batch, hipStream_t stream) {
  dispatch(t, BackwardCall{t, off, param, grad, b, spec, prm, dout, batch, stream});
}

}  // namespace sp::fno
