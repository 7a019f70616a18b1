// Host calls into the engine's interior (see the Makefile).
#include <hip/hip_runtime.h>

#include "blocked.hpp"
#include "blocked_dev.hpp"
#include "engine.hpp"

namespace pysa {
namespace blk {
hipError_t launch_pipe_i8(const BParams& p, int nw, int nt, int groups, hipStream_t st);
hipError_t launch_pipe_bf16_2(const BParams& p, int nw, int nt, int groups, hipStream_t st);
hipError_t launch_pipe_ais_i8(const BParams& p, int nw, int nt, int groups, hipStream_t st);
}  // namespace blk
}  // namespace pysa

// What the launchers of the pipelined kernel answer for nblk blocks: kind 0
// int8, 1 two bf16 pieces, 2 AIS in int8.
extern "C" int probe_launch_pipe(int kind, int order, int nblk, int tiles) {
  pysa::blk::BParams p{};
  p.n = 32 * nblk;
  p.nblk = nblk;
  p.order = order;
  using namespace pysa::blk;
  if (kind == 0) return launch_pipe_i8(p, 4, tiles, 1, nullptr);
  if (kind == 1) return launch_pipe_bf16_2(p, 4, tiles, 1, nullptr);
  return launch_pipe_ais_i8(p, 4, tiles, 1, nullptr);
}

extern "C" int probe_lane_below(int b0, int below) {
  return pysa::blk::lane_below(b0, below);
}

// The plain form's plan (0 a workgroup per read, 1 per chain) on this device.
extern "C" int probe_plan_plain(int n, int reads, int R, int S, int elem, int coupled) {
  return pysa::plan_plain(n, reads, R, S, elem, coupled != 0);
}
