// Two waves that touch the same bytes of LDS between two barriers, one of them writing (compiled without callbacks). Several waves
// may raise one flag of 4 bytes. A request writes its bytes at any time from its issue to the wait that retires it: until the barrier
// after that no other wave may touch them, and its own wave (all lanes issue the same requests and waits) not before the wait; when the
// kernel ends none may be on its way. A block's threads run twice, first for the requests, then for the accesses beside them.
// With LDS_TRACE_NO_BARRIERS set barriers do not count, and every exchange is reported; LDS_TRACE_LAX: so many requests more that a
// wait leaves on their way.
#include <stdlib.h>

#include <algorithm>
#include <deque>
#include <vector>

#include "hip/hip_runtime.h"

dim3 threadIdx, blockIdx, blockDim, gridDim;
float trace_weight;
long long trace_accesses, trace_requests, trace_races;

extern "C" char __start_lds, __stop_lds;  // all __shared__ variables
namespace {
struct Epoch {
  std::vector<unsigned short> read, written;  // the waves, by 4 bytes
};
std::vector<Epoch> epochs;  // by the barriers before
unsigned epoch, event;      // of this thread: barriers; requests and waits
long long low = 1ll << 40, high = -1;  // what was touched
bool checking;

struct Request {
  unsigned wave, from_epoch, to_epoch, from, to;  // from: events before it; to: those before its retirement
};
std::vector<std::vector<Request>> requests;  // by 16 bytes
struct Pending {
  long long at;
  unsigned epoch, event;
};
std::deque<Pending> pending;  // of this thread

int lds_bytes() { return (int)(&__stop_lds - &__start_lds); }

void race(const char* what, unsigned others, long long at) {
  if (++trace_races <= 5)
    printf("block %u, after %u barriers: wave %u %s, waves %x (bits), byte %lld\n", blockIdx.x, epoch, threadIdx.x / 64, what, others, at);
}

void touch(const void* p, int n, bool store) {
  const long long at = (const char*)p - &__start_lds;
  if (!checking || at < 0 || at + n > lds_bytes()) return;
  ++trace_accesses;
  while (epochs.size() <= epoch) epochs.push_back({std::vector<unsigned short>(lds_bytes() / 4 + 1), std::vector<unsigned short>(lds_bytes() / 4 + 1)});
  Epoch& e = epochs[epoch];
  const unsigned wave = threadIdx.x / 64;
  const unsigned short own = 1 << wave;
  low = std::min(low, at / 4), high = std::max(high, (at + n - 1) / 4);
  for (long long g = at / 4; g <= (at + n - 1) / 4; ++g) {
    const unsigned short others = (!store ? e.written[g] : n == 4 ? e.read[g] : e.read[g] | e.written[g]) & ~own;
    if (others) race(store ? "writes what others touch" : "reads what others write", others, g * 4);
    (store ? e.written : e.read)[g] |= own;
  }
  for (long long g = at / 16; g <= (at + n - 1) / 16; ++g)
    for (const Request& r : requests[g])
      if (r.wave == wave ? event >= r.from && event < r.to : epoch >= r.from_epoch && epoch <= r.to_epoch)
        race(store ? "writes what is requested" : "reads what is requested", 1 << r.wave, g * 16);
}

// requests of the same bytes that are on their way at one time
void check_requests() {
  for (size_t g = 0; g < requests.size(); ++g)
    for (size_t i = 0; i < requests[g].size(); ++i)
      for (size_t j = 0; j < i; ++j) {
        const Request &a = requests[g][i], &b = requests[g][j];
        if (a.wave == b.wave ? a.from < b.to && b.from < a.to : a.from_epoch <= b.to_epoch && b.from_epoch <= a.to_epoch)
          race("requests what is requested", 1 << a.wave | 1 << b.wave, g * 16);
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

unsigned lds_offset(const void* p) { return (unsigned)((const char*)p - &__start_lds); }
void lds_request(void* p) { lds_request_at(lds_offset(p)); }
void lds_request_at(unsigned offset) {
  const long long at = offset;
  if (at < 0 || at % 16 || at + 16 > lds_bytes()) abort();
  pending.push_back({at, epoch, ++event});
}

void lds_wait(int newest) {
  static const int lax = getenv("LDS_TRACE_LAX") ? atoi(getenv("LDS_TRACE_LAX")) : 0;
  ++event;
  while ((int)pending.size() > newest + lax) {
    const Pending& r = pending.front();
    if (!checking) requests[r.at / 16].push_back({threadIdx.x / 64, r.epoch, epoch, r.event, event}), ++trace_requests;
    pending.pop_front();
  }
}

// The first blocks of the grid and the last one
void run(dim3 grid, dim3 block, void (*thread)(void*), void* what) {
  gridDim = grid, blockDim = block;
  for (blockIdx.x = 0; blockIdx.x < grid.x; ++blockIdx.x) {
    if (blockIdx.x >= 4 && blockIdx.x + 1 < grid.x) continue;
    for (Epoch& e : epochs)
      for (auto* v : {&e.read, &e.written}) std::fill(v->begin() + low, v->begin() + high + 1, 0);
    requests.assign(lds_bytes() / 16 + 1, {});
    for (bool second : {false, true}) {
      checking = second;
      for (threadIdx.x = 0; threadIdx.x < block.x; ++threadIdx.x) {
        epoch = event = 0;
        thread(what);
        if (!second && !pending.empty()) race("ends with requests on their way", 1 << threadIdx.x / 64, pending.front().at);
        pending.clear();
      }
      if (!second) check_requests();
    }
  }
}
