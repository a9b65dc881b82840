// Host launchers of the stage kernels, shared by the workspace and the pass-level
// entry points. Each enqueues one kernel on `s`; none synchronises.
#pragma once

#include "device.hpp"

namespace sp {

// What the envelope route's stage kernels (env_stage.hip) work on. The fine grid's T = n1 n2
// samples (n2 = n1 or 2 n1) are split one way and the other in turn, so the kernels read
// `in` and write `out` in layouts of their own between them: the entry and finish leave
// what the drive (with Raman, else the response) reads, and so on round the stage.
struct EnvStage {
  DeviceProblem P;
  const TrialRecord* R;
  const cplx* in;   // T points, and a second row of the in-stage absorber's term
  cplx* out;
  cplx* field;      // the stage's time samples, from the drive to the response
  cplx *y, *k, *einv, *adv, *recycled;  // (N), k (n_stages, N)
  double* partials;                     // 3 rows of env_accept_blocks
  const cplx* roots;       // W_T^t, t < T
  const cplx* roots_l[2];  // W_n1, W_n2
  const cplx* twist;       // W_4T^t, t < T
  const cplx* kernel;      // the transform of the Raman response (launch_env_raman_kernel)
  int log2n1, log2n2;
  int commit, recycle;  // the entry first commits `adv` into y (band mask), copies recycled to k[0]
};

unsigned env_accept_blocks(const EnvStage& a);
// The Raman response at `stage`'s rates as w (h1 + i h2) into `z` (T points), to be
// transformed forward into EnvStage::kernel.
void launch_env_raman_kernel(const EnvStage& a, int stage, cplx* z, hipStream_t s);
void launch_env_entry(const EnvStage& a, int stage, hipStream_t s);
void launch_env_drive(const EnvStage& a, int stage, hipStream_t s);
void launch_env_product(const EnvStage& a, int stage, hipStream_t s);
void launch_env_response(const EnvStage& a, int stage, hipStream_t s);
// Stage `stage - 1`'s finish and stage `stage`'s entry (stage >= 1).
void launch_env_finish(const EnvStage& a, int stage, hipStream_t s);
// The last stage's finish and the step's acceptance.
void launch_env_accept(const EnvStage& a, hipStream_t s);

// Over `rows` consecutive rows of T packed points, one kernel spectrum for all.
void launch_raman_product(cplx* z, const cplx* H, const cplx* roots2T, int T, int rows,
                          hipStream_t s);
void launch_raman_kernel_post(const cplx* z, cplx* H, const cplx* roots2T, int T, double dt,
                              hipStream_t s);
// The upload of `bytes` (whole doubles) from pinned host memory (`host` as the device
// addresses it) to `device`, as a kernel of one workgroup that reads them at system scope.
void launch_record_fetch(const void* host, void* device, std::size_t bytes, hipStream_t s);
void launch_commit_masked(const DeviceProblem& P, const cplx* adv, cplx* y, hipStream_t s);
void launch_copy_points(const cplx* src, cplx* dst, long n, hipStream_t s);
// The envelope route's split-step absorber, around the caller's inverse and forward
// transforms of the coarse grid (the unpack is `launch_commit_masked` from the buffer).
void launch_env_split_pack(const DeviceProblem& P, const cplx* y, cplx* buf, hipStream_t s);
void launch_env_split_collar(const DeviceProblem& P, const TrialRecord* R, double dz, cplx* buf,
                             hipStream_t s);

}  // namespace sp
