// The expert tiles' own source for the host, every load and store with a callback (trace.cpp). Arguments: "stream", "block" or "turns", 1 for gate
// and up, rows, stages of 64 of K. Or "once": which tiles' weights come non-temporal, for experts of any number of rows.
#include <stdlib.h>

#include <initializer_list>

#include "../../csrc/kernels/expert_tiles.h"

extern long long trace_accesses, trace_requests, trace_races;

template <bool UP, int XI>
void stream(ExpertArgs p, int rows) {
  __shared__ __attribute__((aligned(1024))) char sl[STREAM_LDS];
  expert_stream_tile<UP, XI>(p, sl, 0, 0, rows, 16);
}
template <bool UP>
void block(ExpertArgs p, int rows) {
  __shared__ __attribute__((aligned(1024))) char sl[STREAM_LDS];
  expert_block_tile<UP>(p, sl, 0, 0, rows, 0);
}
template <bool UP, int B>
void turns(ExpertArgs p, int rows) {
  __shared__ __attribute__((aligned(1024))) char sl[WIDE_LDS];
  expert_turns_tile<UP, B>(p, sl, 0, 0, rows, 0);
}

template <bool UP>
void tile(char form, const ExpertArgs& p, int rows) {
  auto go = [&](auto f, int threads) { hipLaunchKernelGGL(f, dim3(1), dim3(threads), 0, nullptr, p, rows); };
  if (form == 't') rows > 192 ? go(turns<UP, 4>, 512) : rows > 128 ? go(turns<UP, 3>, 512) : rows > 64 ? go(turns<UP, 2>, 512) : go(turns<UP, 1>, 512);
  else if (form == 'b') go(block<UP>, 256);
  else rows > 16 ? go(stream<UP, 4>, 256) : rows > 8 ? go(stream<UP, 2>, 256) : go(stream<UP, 1>, 256);
}

// An expert's c rows: full tiles side by side, and the rest, among them or after all others. Weights that are read again come through the cache.
int once() {
  int wrong = 0, seen = 0;
  for (int mt : {128, 192})
    for (int c = 1; c < 1000; ++c) {
      const int late = late_tile(c, mt), beside = (c + mt - 1) / mt - late;
      for (int i = 0; i < beside; ++i) {
        const bool is = read_once(beside, c - i * mt < mt ? c - i * mt : mt, mt);
        wrong += is && (beside > 1 || late), seen += is;
      }
      seen += late && read_once(1, c % mt, mt);
    }
  printf("wrong %d\nonce %d\n", wrong, seen);
  return 0;
}

int main(int argc, char** argv) {
  if (argc == 2) return once();
  if (argc != 5) return 2;
  const int rows = atoi(argv[3]), N = 48;
  int* perm = (int*)calloc(rows, 4);
  for (int i = 0; i < rows; ++i) perm[i] = i;
  ExpertArgs p{};
  p.perm = perm, p.wts = (float*)calloc(rows, 4), p.y = calloc(rows * N, 2), p.top = 1, p.N = N, p.K = 64 * atoi(argv[4]), p.scale = 1;
  if (atoi(argv[2])) tile<true>(argv[1][0], p, rows);
  else tile<false>(argv[1][0], p, rows);
  printf("accesses %lld\nrequests %lld\nraces %lld\n", trace_accesses, trace_requests, trace_races);
  return 0;
}
