// The one-launch z-loop (loop.hpp) for rows of 128 points.
#include "loop.hpp"

bool bpmh_loop_nx128(int ny, int er, int ec, int mode, const LoopCall& c, int groups, hipStream_t s) {
  return loop_launch_nx<128>(ny, er, ec, mode, c, groups, s);
}
