// The attention kernels' own source for the host, every load and store with a callback (trace.cpp). Arguments: "fwd" or "bwd", head
// size, batch, queries, keys, heads, KV heads, window, ALiBi, lengths, weight (a large one: every row's sum overflows).
#include <stdlib.h>

#include "../../csrc/kernels/attention_split.hip"
#include "../../csrc/kernels/attention_pair.hip"

extern long long trace_accesses, trace_requests, trace_races;

int main(int argc, char** argv) {
  if (argc != 12) return 2;
  auto arg = [&](int i) { return atoi(argv[i]); };
  const int D = arg(2), B = arg(3), Sq = arg(4), Sk = arg(5), H = arg(6), Hkv = arg(7);
  trace_weight = (float)atof(argv[11]);
  const long long qt = (long long)H * D, kt = (long long)Hkv * D;
  auto rows = [&](long long st, int S) { return (bf16_t*)calloc(B * S * st, 2); };
  auto stat = [&] { return (float*)calloc(B * H * Sq, 4); };
  float* slopes = stat();
  int* lens = (int*)calloc(B, 4);
  for (int b = 0; b < B; ++b) lens[b] = max(0, Sk - 37 * b);
  auto common = [&](auto& p) {
    p.q = rows(qt, Sq), p.k = rows(kt, Sk), p.v = rows(kt, Sk), p.o = rows(qt, Sq), p.lse = stat();
    p.q_sb = p.o_sb = Sq * qt, p.k_sb = p.v_sb = Sk * kt, p.q_st = p.o_st = qt, p.k_st = p.v_st = kt, p.q_sh = p.k_sh = p.v_sh = p.o_sh = D;
    p.B = B, p.Sq = Sq, p.Sk = Sk, p.H = H, p.Hkv = Hkv, p.scale = 0.1f, p.window = arg(8);
    p.alibi = arg(9) ? slopes : nullptr, p.kv_len = arg(10) ? lens : nullptr;
  };
  int rc;
  if (argv[1][0] == 'f') {
    FastFwdParams p{};
    common(p);
    rc = attn_fwd_split(p, D, nullptr);
  } else {
    FastBwdParams p{};
    common(p);
    p.dout = rows(qt, Sq), p.dq = rows(qt, Sq), p.dk = rows(kt, Sk), p.dv = rows(kt, Sk), p.delta = stat();
    p.do_sb = p.dq_sb = p.q_sb, p.dk_sb = p.dv_sb = p.k_sb, p.do_st = p.dq_st = qt, p.dk_st = p.dv_st = kt;
    p.do_sh = p.dq_sh = p.dk_sh = p.dv_sh = D;
    rc = D == 256 ? attn_bwd_pair(p, D, true, nullptr) : attn_bwd_split(p, D, nullptr);
  }
  printf("accesses %lld\nrequests %lld\nraces %lld\n", trace_accesses, trace_requests, trace_races);
  return rc;
}
