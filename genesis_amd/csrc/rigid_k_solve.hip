// Newton solve of the plain step: k_solve (one lane per env), or on wavefronts k_solve_dense (every dof in one entity),
// k_solve_bodies<2 | 4> (free bodies, two or four wavefronts per env) or k_solve_wave (entity blocks).
#include "rigid_tiles.h"

namespace gsr {
namespace {

__global__ void __launch_bounds__(kBlock) k_solve(gsr_model m, gsr_state s) {
  int b = env_id();
  if (b >= s.n_envs) return;
  Env e(m, s, b);
  dev_solve(e);
}

__global__ void __launch_bounds__(kWave) k_solve_wave(gsr_model m, gsr_state s) {
  extern __shared__ char lds[];
  if ((int)blockIdx.x >= s.n_envs) return;  // uniform across the block
  const int b = xcd_env(blockIdx.x, s.n_envs);
  Env e(m, s, b);
  wave_solve_blocks(e, lds);
}

// the single-entity solver alone: it takes about half the registers of the entity-block solver, so a SIMD holds more envs
__global__ void __launch_bounds__(kWave) k_solve_dense(gsr_model m, gsr_state s) {
  extern __shared__ char lds[];
  if ((int)blockIdx.x >= s.n_envs) return;  // uniform across the block
  const int b = xcd_env(blockIdx.x, s.n_envs);
  Env e(m, s, b);
  wave_solve_dense(e, lds);
}

// Free bodies, kWaves wavefronts per env. Left to itself the compiler takes 250 VGPRs (two waves a SIMD); held to three
// waves (168) for two wavefronts an env and to four (128) for four it spills to scratch but hides more latency: 1,500
// 20-box piles 3,758 -> 3,318 us a pass, 4,096 64-box piles 32,383 -> 25,206 us (two, three, four: 32.9, 27.7, 25.2 ms).
template <int kWaves>
__global__ void __launch_bounds__(kWave * kWaves) __attribute__((amdgpu_waves_per_eu(kWaves == 2 ? 3 : 4))) k_solve_bodies(gsr_model m, gsr_state s) {
  extern __shared__ char lds[];
  if ((int)blockIdx.x >= s.n_envs) return;  // uniform across the block
  const int b = xcd_env(blockIdx.x, s.n_envs);
  Env e(m, s, b);
  solve_bodies<kWaves>(e, lds);
}

}  // namespace

void launch_solve(const gsr_model& m, const gsr_state& s, hipStream_t st) {
  const size_t lds = solve_lds_bytes(m);
  switch (solve_form(m)) {
    case kSolveLane: hipLaunchKernelGGL(k_solve, dim3((s.n_envs + kBlock - 1) / kBlock), dim3(kBlock), 0, st, m, s); break;
    case kSolveDense: hipLaunchKernelGGL(k_solve_dense, dim3(s.n_envs), dim3(kWave), lds, st, m, s); break;
    case kSolveBodies2: hipLaunchKernelGGL(k_solve_bodies<2>, dim3(s.n_envs), dim3(2 * kWave), lds, st, m, s); break;
    case kSolveBodies4: hipLaunchKernelGGL(k_solve_bodies<4>, dim3(s.n_envs), dim3(4 * kWave), lds, st, m, s); break;
    case kSolveBlocks: hipLaunchKernelGGL(k_solve_wave, dim3(s.n_envs), dim3(kWave), lds, st, m, s); break;
  }
}

}  // namespace gsr
