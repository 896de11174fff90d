// block_of for the host: every block of every head once, whatever the sizes.
#include <vector>

#include "../../csrc/kernels/attn_fast.h"

dim3 threadIdx, blockIdx, blockDim, gridDim;
float trace_weight;
void barrier() {}
void run(dim3, dim3, void (*)(void*), void*) {}

template <bool CAUSAL, int D, int ROWS, int PER_CU>
int check() {
  int bad = 0;
  for (int blocks : {1, 2, 3, 4, 5, 7, 8, 9, 12, 16, 31})
    for (int heads : {1, 3, 7, 8, 9, 16, 20, 64, 129, 180, 640, 1280}) {
      gridDim.x = blocks * heads;
      std::vector<char> seen(gridDim.x);
      for (blockIdx.x = 0; blockIdx.x < gridDim.x; ++blockIdx.x) {
        const BlockOf b = block_of<CAUSAL, D, ROWS, PER_CU>(blocks, heads);
        if (b.block < 0 || b.block >= blocks || b.head < 0 || b.head >= heads || seen[b.head * blocks + b.block]++) ++bad;
      }
      if (bad) printf("D %d, rows %d: %d blocks of %d heads: %d\n", D, ROWS, blocks, heads, bad);
    }
  return bad;
}

int main() {
  return check<true, 64, 64, 3>() + check<true, 64, 128, 3>() + check<true, 96, 64, 1>() + check<true, 96, 128, 1>() + check<true, 96, 128, 3>() + check<true, 160, 128, 1>() + check<true, 128, 128, 1>() +
         check<true, 256, 128, 1>() + check<true, 256, 256, 1>() + check<false, 64, 128, 1>() != 0;
}
