// The pipelined tile GEMM (gemm_pipe.hip) with the K chunks of a tile in workgroups of their own.
#include "gemm_pipe_tile.h"

int gemm_pipe_split(const GemmSkCall& p, int layout, hipStream_t st) { return gp_layout<false, true>(p, layout, st); }
