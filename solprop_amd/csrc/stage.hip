// Pointwise kernels of the envelope workspace and the Raman product of the field routes,
// FP64, for gfx950 (the envelope's stages are in env_stage.hip).
#include "kernels.hpp"

namespace sp {

namespace {

__device__ inline cplx r2c_post(cplx za, cplx zb, cplx w) {
  // X = E + W O with E = (Za + conj Zb)/2, O = -i (Za - conj Zb)/2.
  const cplx e = scale(0.5, add(za, conj(zb)));
  const cplx o = scale(0.5, rot(sub(za, conj(zb)), -1));
  return add(e, mul(w, o));
}

}  // namespace

// One pair (k, T-k) of the packed doubled-grid transform of row blockIdx.y: unpack the
// real transform, multiply by the kernel spectrum, and pack again for the inverse, in
// place.
__global__ void raman_product(cplx* z, const cplx* H, const cplx* roots2T, int T) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k > T / 2) return;
  z += static_cast<long>(blockIdx.y) * T;
  const int kk = (T - k) % T;
  const cplx za = z[k], zb = z[kk];
  const cplx xa = r2c_post(za, zb, roots2T[k]);
  const cplx xb = r2c_post(zb, za, roots2T[T - k]);
  const cplx ya = mul(H[k], xa), yb = mul(H[T - k], xb);
  z[k] = c2r_pre(ya, yb, roots2T[k]);
  if (k > 0 && k != T - k) z[T - k] = c2r_pre(yb, ya, roots2T[T - k]);
}

// H[k] = rfft(h)[k] dt for k in [0, T].
__global__ void raman_kernel_post(const cplx* z, cplx* H, const cplx* roots2T, int T,
                                  double dt) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k > T) return;
  const cplx x = r2c_post(z[k % T], z[(T - k) % T], roots2T[k]);
  H[k] = scale(dt, x);
}

__global__ void commit_masked(DeviceProblem P, const cplx* adv, cplx* y) {
  const long idx = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
  const long CN = static_cast<long>(P.C) * P.N;
  if (idx >= CN) return;
  y[idx] = P.active[idx % P.N] ? adv[idx] : make(0.0, 0.0);
}

// The split-step absorber on the committed envelope (the workspace's finish,
// src/solprop/backends/numpy_ref/workspace.py:1021-1106): the masked state to time
// samples (1/N folded in before the unscaled inverse transform), times exp(-alpha h / 2)
// with h the accepted step (the record's, inside a graph; else `dz`), and, after the
// forward transform, back onto the state with the band imposed again.
__global__ void env_split_pack(DeviceProblem P, const cplx* y, cplx* buf) {
  const long idx = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (idx >= static_cast<long>(P.C) * P.N) return;
  buf[idx] = scale(1.0 / P.N, y[idx]);
}

__global__ void env_split_collar(DeviceProblem P, const TrialRecord* R, double dz, cplx* buf) {
  const long idx = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (idx >= static_cast<long>(P.C) * P.N) return;
  const double h = R ? R->accepted_dz : dz;
  buf[idx] = scale(exp((-0.5 * P.absorber_rate[idx % P.N]) * h), buf[idx]);
}

__global__ void copy_points(const cplx* src, cplx* dst, long n) {
  const long idx = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (idx < n) dst[idx] = src[idx];
}

// -------------------------------------------------------------------- launchers

namespace {
constexpr int kThreads = 256;
void check_launch() { SP_HIP(hipGetLastError()); }
}  // namespace

void launch_raman_product(cplx* z, const cplx* H, const cplx* roots2T, int T, int rows,
                          hipStream_t s) {
  hipLaunchKernelGGL(raman_product, dim3(blocks_for(T / 2 + 1, kThreads), rows),
                     dim3(kThreads), 0, s, z, H, roots2T, T);
  check_launch();
}

void launch_raman_kernel_post(const cplx* z, cplx* H, const cplx* roots2T, int T, double dt,
                              hipStream_t s) {
  hipLaunchKernelGGL(raman_kernel_post, dim3(blocks_for(T + 1, kThreads)), dim3(kThreads), 0,
                     s, z, H, roots2T, T, dt);
  check_launch();
}

void launch_commit_masked(const DeviceProblem& P, const cplx* adv, cplx* y, hipStream_t s) {
  const std::size_t n = static_cast<std::size_t>(P.C) * P.N;
  hipLaunchKernelGGL(commit_masked, dim3(blocks_for(n, kThreads)), dim3(kThreads), 0, s, P, adv,
                     y);
  check_launch();
}

void launch_env_split_pack(const DeviceProblem& P, const cplx* y, cplx* buf, hipStream_t s) {
  const std::size_t n = static_cast<std::size_t>(P.C) * P.N;
  hipLaunchKernelGGL(env_split_pack, dim3((n + kThreads - 1) / kThreads), dim3(kThreads), 0, s,
                     P, y, buf);
  check_launch();
}

void launch_env_split_collar(const DeviceProblem& P, const TrialRecord* R, double dz, cplx* buf,
                             hipStream_t s) {
  SP_CHECK(P.absorber_rate, "the split-step absorber's rate");
  const std::size_t n = static_cast<std::size_t>(P.C) * P.N;
  hipLaunchKernelGGL(env_split_collar, dim3((n + kThreads - 1) / kThreads), dim3(kThreads), 0,
                     s, P, R, dz, buf);
  check_launch();
}

void launch_copy_points(const cplx* src, cplx* dst, long n, hipStream_t s) {
  hipLaunchKernelGGL(copy_points, dim3(blocks_for(static_cast<std::size_t>(n), kThreads)),
                     dim3(kThreads), 0, s, src, dst, n);
  check_launch();
}

}  // namespace sp
