// The surrogate's fused tile path: one kernel a Fourier layer in each direction, for
// networks of at most 64 channels, 64 retained modes and 128 head units.
//
// A workgroup owns one sample and a run of 64-point column tiles. Per tile it forms the
// layer's output in registers (the 1x1 convolution and the inverse truncated transform in
// one contraction), applies the activation, hands the tile over through LDS, and from
// there both stores it and contracts it with the next forward transform, whose
// (modes x channels) sum stays in registers over the run. The backward layer does the same
// with the gradient, recomputing the pre-activation instead of having stored it.
#pragma once

#include <hip/hip_runtime.h>

#include <vector>

#include "fno.hpp"

namespace sp::fno {

constexpr int kTile = 64;       // columns a tile
constexpr int kHeadUnits = 128; // the head's padded width

// Padded sizes of a network the tile path runs.
struct TileShape {
  int W, M, H, n, np;  // channels, modes, head units, bins, scan parameters
  int WP, MP, NP;      // channels padded to 32 or 64, 2 modes padded to 64 or 128, bins to 64
};

// Whether the tile path runs this network, and its padded shape.
bool tile_available(const Shape& s);
TileShape tile_shape(const Shape& s);

// How a batch's column tiles split over workgroups: `per` tiles a workgroup, `chunks`
// workgroups a sample.
struct TileSplit {
  int per, chunks;
};

// One partial-sum output of the weight gradients: `rows` x `cols` values at
// src + workgroup * stride (leading dimension src_ld), summed over the workgroups into dst
// (leading dimension dst_ld). With `scan_parameter` >= 0 each workgroup's value is weighted
// by that scan parameter of its sample.
struct GradientSegment {
  const float* src;
  long stride;
  float* dst;
  int rows, cols, src_ld, dst_ld, scan_parameter, first_block;
};

// Device memory of the tile path (allocated by the network that owns it).
struct TileBuffers {
  // Transform tables: `_s` rows are bins (modes contiguous), `_k` rows modes.
  bf16 *g_s, *f_k, *f_s, *g_k;
  // Padded parameters, per layer: the convolution and its transpose; the head's and its
  // transpose.
  std::vector<bf16*> w, wt;
  bf16 *q1, *q1t;
  std::vector<bf16*> v;       // activations (B, NP, WP), layers + 1
  // Spectra: (MP, rows, WP) with `rows` the most samples a batch has, so that the rows of
  // the padded modes are never written and stay zero.
  int rows;
  std::vector<bf16*> yhat;    // mixed, a layer
  bf16* dvhat;
  std::vector<float*> vhat;   // summed (MP, B, WP), a layer
  std::vector<float*> dyhat;  // their gradients
  bf16* dz[2];                // (B, NP, WP)
  float* share;               // a workgroup's spectral sums: (chunks, MP, B, WP)
  std::vector<float*> dw;     // per workgroup: WP x WP, then WP bias sums; a layer
  float* dq;                  // per workgroup: H' x WP, then H' bias, H' and 1 output sums
  float* dlift;               // per workgroup: 3 x WP
  float* loss;                // per workgroup
  GradientSegment* segments;
  int n_segments, segment_blocks;
};

// Floats of a workgroup's share of the head's sums.
constexpr long head_share(int WP) {
  return static_cast<long>(kHeadUnits) * WP + 2 * kHeadUnits + WP + 1;
}

TileSplit tile_split(const TileShape& t, int batch, int workgroups);
// Workgroups a launch aims at in each direction, and the most a batch of at most
// `max_batch` samples takes.
constexpr int kForwardGroups = 512, kBackwardGroups = 256;
long tile_groups(int max_batch);

// The parameters' padded copies (after they change).
void tile_pack(const TileShape& t, const Offsets& off, const float* param, const TileBuffers& b,
               hipStream_t stream);
// The output (B, n); with `target` also dout = 2 (out - target) / (B n) and the mean
// squared error in *loss. `keep` stores what the gradient needs.
void tile_forward(const TileShape& t, const Offsets& off, const float* param,
                  const TileBuffers& b, const float* spec, const float* prm, float* out,
                  const float* target, float* dout, float* loss, int batch, bool keep,
                  hipStream_t stream);
// The gradient of every parameter from dout, after a kept forward pass of the same batch.
void tile_backward(const TileShape& t, const Offsets& off, const float* param, float* grad,
                   const TileBuffers& b, const float* spec, const float* prm, const float* dout,
                   int batch, hipStream_t stream);

}  // namespace sp::fno
