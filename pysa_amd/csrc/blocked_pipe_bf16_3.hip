// Pipelined MFMA kernel, 3 bf16 pieces.
#include "blocked_pipe.hpp"

namespace pysa {
namespace blk {

hipError_t launch_pipe_bf16_3(const BParams& p, int nw, int nt, int groups, hipStream_t st) {
  return launch_pipe_enc<3, false>(p, nw, nt, groups, st);
}

hipError_t launch_pipe_ais_bf16_3(const BParams& p, int nw, int nt, int groups, hipStream_t st) {
  return launch_pipe_ais_enc<3, false>(p, nw, nt, groups, st);
}

}  // namespace blk
}  // namespace pysa
