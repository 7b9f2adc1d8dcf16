// The one-launch adjoint z-loop (loop_adj.hpp) for rows of 512 points.
#include "loop_adj.hpp"

bool bpmh_loop_adj_nx512(int ny, int er, int ec, int mode, const LoopCall& c, int groups, hipStream_t s) {
  return loop_adj_launch_nx<512>(ny, er, ec, mode, c, groups, s);
}
