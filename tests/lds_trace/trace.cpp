// Two waves that touch the same bytes of LDS between two barriers, one of them writing (compiled without callbacks). Several waves
// may raise one flag of 4 bytes. With LDS_TRACE_NO_BARRIERS set barriers do not count, and every exchange is reported.
#include <stdlib.h>

#include <algorithm>
#include <vector>

#include "hip/hip_runtime.h"

dim3 threadIdx, blockIdx, blockDim, gridDim;
float trace_weight;
long long trace_accesses, trace_races;

extern "C" char __start_lds, __stop_lds;  // all __shared__ variables
namespace {
struct Epoch {
  std::vector<unsigned short> read, written;  // the waves, by 4 bytes
};
std::vector<Epoch> epochs;  // by the barriers before
unsigned epoch;
long long low = 1ll << 40, high = -1;  // what was touched

void touch(const void* p, int n, bool store) {
  const int bytes = (int)(&__stop_lds - &__start_lds);
  const long long at = (const char*)p - &__start_lds;
  if (at < 0 || at + n > bytes) return;
  ++trace_accesses;
  while (epochs.size() <= epoch) epochs.push_back({std::vector<unsigned short>(bytes / 4 + 1), std::vector<unsigned short>(bytes / 4 + 1)});
  Epoch& e = epochs[epoch];
  const unsigned short own = 1 << (threadIdx.x / 64);
  low = std::min(low, at / 4), high = std::max(high, (at + n - 1) / 4);
  for (long long g = at / 4; g <= (at + n - 1) / 4; ++g) {
    const unsigned short others = (!store ? e.written[g] : n == 4 ? e.read[g] : e.read[g] | e.written[g]) & ~own;
    if (others && ++trace_races <= 5)
      printf("block %u, after %u barriers: wave %u %s what waves %x (bits) touch, byte %lld\n", blockIdx.x, epoch, threadIdx.x / 64,
             store ? "writes" : "reads", others, g * 4);
    (store ? e.written : e.read)[g] |= own;
  }
}
}  // namespace

extern "C" {
#define CALLBACKS(N)                                            \
  void __sanitizer_cov_load##N(void* p) { touch(p, N, false); } \
  void __sanitizer_cov_store##N(void* p) { touch(p, N, true); }
CALLBACKS(1) CALLBACKS(2) CALLBACKS(4) CALLBACKS(8) CALLBACKS(16)
void __sanitizer_cov_trace_pc() {}
}

void barrier() {
  static const bool count = !getenv("LDS_TRACE_NO_BARRIERS");
  epoch += count;
}

// The first blocks of the grid and the last one
void run(dim3 grid, dim3 block, void (*thread)(void*), void* what) {
  gridDim = grid, blockDim = block;
  for (blockIdx.x = 0; blockIdx.x < grid.x; ++blockIdx.x) {
    if (blockIdx.x >= 4 && blockIdx.x + 1 < grid.x) continue;
    for (Epoch& e : epochs)
      for (auto* v : {&e.read, &e.written}) std::fill(v->begin() + low, v->begin() + high + 1, 0);
    for (threadIdx.x = 0; threadIdx.x < block.x; ++threadIdx.x) {
      epoch = 0;
      thread(what);
    }
  }
}
