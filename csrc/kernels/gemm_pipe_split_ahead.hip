// The pipelined tile GEMM (gemm_pipe.hip) with K chunks and with workgroups that touch later weights.
#include "gemm_pipe_tile.h"

int gemm_pipe_split_ahead(const GemmSkCall& p, int layout, hipStream_t st) { return gp_layout<true, true>(p, layout, st); }
