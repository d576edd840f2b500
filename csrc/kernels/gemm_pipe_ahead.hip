// The pipelined tile GEMM (gemm_pipe.hip) with workgroups behind the tiles' that touch the weights
// of later launches.
#include "gemm_pipe_tile.h"

int gemm_pipe_ahead(const GemmSkCall& p, int layout, hipStream_t st) { return gp_layout<true, false>(p, layout, st); }
