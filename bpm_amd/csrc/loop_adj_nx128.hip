// The one-launch adjoint z-loop (loop_adj.hpp) for rows of 128 points.
#include "loop_adj.hpp"

bool bpmh_loop_adj_nx128(int ny, int er, int ec, int mode, const LoopCall& c, int groups, hipStream_t s) {
  return loop_adj_launch_nx<128>(ny, er, ec, mode, c, groups, s);
}
