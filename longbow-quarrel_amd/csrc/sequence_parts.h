// A step's sequences in parts of up to `size` rows (tiles, chunks), numbered through the sequences: which part a workgroup
// takes.
#pragma once

#include "common.h"

namespace {

// The parts of a sequence of n rows: none for one shorter than `least`.
__device__ inline int parts_of(int n, int size, int least) { return n >= least ? (n + size - 1) / size : 0; }

struct Part {
  int seq, number, first, rows;  // the sequence (-1: past the last part), the part's number within it, its first row and rows
};

// Part number t.  Lane i holds sequence i of a run of 64; every wavefront works out the same.
__device__ inline Part find_part(const int* __restrict__ cu_rows, int batch, int size, int least, int t) {
  const int lane = threadIdx.x & 63;
  for (int b0 = 0; b0 < batch; b0 += 64) {
    const int b = min(b0 + lane, batch - 1), begin = cu_rows[b], n = b0 + lane < batch ? cu_rows[b + 1] - begin : 0;
    const int mine = b0 + lane < batch ? parts_of(n, size, least) : 0;
    int upto = mine;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int before = __shfl_up(upto, off, 64);
      if (lane >= off) upto += before;
    }
    const unsigned long long past = __ballot(upto > t);
    if (past) {
      const int at = __ffsll(past) - 1, k = t - __shfl(upto - mine, at, 64);
      const int first = __shfl(begin, at, 64) + k * size, rows = min(size, __shfl(n, at, 64) - k * size);
      return {__builtin_amdgcn_readfirstlane(b0 + at), __builtin_amdgcn_readfirstlane(k), __builtin_amdgcn_readfirstlane(first),
              __builtin_amdgcn_readfirstlane(rows)};
    }
    t -= __shfl(upto, 63, 64);
  }
  return {-1, -1, 0, 0};
}

}  // namespace
