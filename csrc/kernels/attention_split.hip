// Flash attention, causal calls of 64, 96 and 128 wide heads with 16-byte rows: blocks of 128 rows and four waves, or, where those leave the
// chip idle, of 64 rows whose keys (dK/dV: queries) are split over two groups of waves. (Full tiles of 64-wide heads in many blocks stay with
// attention_tiled.hip's plain forms: kca_attn_fwd_tiled, kca_attn_bwd_tiled.)
//
// What bounds these calls. A block of 128 rows gives a wave 32 of them; a call of few heads and rows then has less than one
// workgroup a CU, so a SIMD runs one wave whose products, softmax, LDS reads and barriers follow
// each other, and under a causal mask the call waits for the block that sees all keys: 2048 tokens x 14 heads of 128 are 224
// workgroups on 256 CUs, 52 us for the 64 tiles of the longest one. Here a workgroup has RW * 32 rows and KG groups of RW
// waves; group g walks tiles g, g + KG, ... with LDS buffers of its own and the partial sums meet in LDS at the end. Two groups'
// blocks are half as tall, so there are twice as many, each half as long, and a SIMD has two waves to run. Many blocks gain from
// one group too: overflowed rows take no launch of their own, and blocks go longest first.
//
// The forms of a mask are attention_tiled.hip's general ones (1: lengths, windows, any sizes; 2: ALiBi) and every call takes
// one of them. The order of the blocks: block_of.
//
// Tiles go from memory straight into LDS (TileRequests), NB of K and NB of V a group in turn: three steps ahead of their use with one group, one
// or two where two groups' tiles fill the LDS. One barrier a step: behind it a tile has landed for all waves and another has been read by all,
// whose place is requested at once. A wave requests K or V, not both; a request of 1 KB takes a CU's address path 16 cycles, so those of
// a step stand between its products. What it replaces, tiles through registers one step ahead, cost their LDS stores, 16 registers and, at a
// step's end, the wait for memory: a step of 96-wide rows took 1300 cycles alone on its CU, now 1000 (384 of products), and 168
// registers let a third workgroup run. The forward computes S of the next tile while it takes the softmax of this one, so it reads K a tile ahead.
// us, before and now: forward 1 x 1500 x 64 x 96 58 -> 48, 4 x 2048 x 32 x 96 160 -> 133, 2 x 2048 x 20 x 128 60 -> 54, 1 x 4000 x 20 x 128 105 -> 91, 3 x 2048
// x 16 x 64 40.5 -> 38; backward 1 x 1500 x 64 x 96 144 -> 136, 2 x 2048 x 20 x 128 190 -> 169, 2048 x 14 x 128 with ALiBi 112 -> 95,
// 4 x 2048 x 32 x 96 436 -> 407, 8 x 1000 x 12 x 64 72 -> 71. (The forward's scores are no longer copied from step to step: 3 % of it.)
//
// Softmax reference: as in attn_fwd_tiled_kernel the row's maximum over the first tile with a visible key, here of each
// group; the groups' sums are scaled to the largest reference when they meet. Rows whose sum passes 2^100 (a later score far
// above the first tile's) are computed again in the same launch with the row's true maximum.
#include "attn_fast.h"

#include <type_traits>

namespace {

constexpr int kNoTile = 1 << 29;  // first "key" of a tile past the end of a group's walk: masks everything

template <int D, int G, int RW, int KG, int WPS>
__global__ void __launch_bounds__(64 * RW * KG, WPS) attn_fwd_split_kernel(FastFwdParams p) {
  constexpr int BM = 32 * RW, BN = 32;
  constexpr int TILE = BN * D * 2, KS = D / 16;
  constexpr int NB = KG == 1 ? 4 : D == 128 ? 2 : 3;  // tiles of K and of V in LDS, a group
  using Req = TileRequests<D, RW / 2>;                // (half of a group's waves request K, the others V)
  constexpr int PART = 32 * D * 4;  // a wave's partial sums
  static_assert((KG - 1) * RW * PART <= KG * 2 * NB * TILE, "the partial sums take the tiles' place");
  __shared__ __attribute__((aligned(16))) char smem[KG * 2 * NB * TILE];  // per group [K's NB tiles | V's]
  __shared__ float stat[KG][RW][32][2];                              // reference, sum of each row and group
  __shared__ int again;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = wave / RW, rw = wave % RW;
  const int l32 = lane & 31, hh = lane >> 5, gi = lane & 15;
  const int nqb = (p.Sq + BM - 1) / BM, heads = p.B * p.H;
  const auto [qi, bh] = block_of<true, D, BM, WPS == 3 ? 3 : 1>(nqb, heads);
  const int qb = nqb - 1 - qi;
  const int b = bh / p.H, h = bh % p.H;
  const int hk = h / (p.H / p.Hkv);
  if (p.cu) {
    own_sequence(p, b);
    if (qb * BM >= p.Sq) return;
  }
  const int off = p.Sk - p.Sq;
  const int q0 = qb * BM + rw * 32, qrow = q0 + l32;
  const int kv_end = batch_keys(p.kv_len, b, p.Sk);
  const TileSpan sp = tile_span<BM, true, G == 1 ? 2 : 0>(qb * BM, off, kv_end, p.window);
  const int ntiles = sp.hi - sp.lo, nsteps = (ntiles + KG - 1) / KG;
  auto index = [&](int i) { return KG * i + g; };                      // the group's i-th tile, counted along the walk
  auto key0 = [&](int i) {                                             // its first key
    const int n = min(index(i), ntiles - 1);
    return (G == 2 ? sp.hi - 1 - n : sp.lo + n) * BN;
  };
  auto mkey0 = [&](int i) { return index(i) < ntiles ? key0(i) : kNoTile; };  // as the mask sees it
  const float sl2 = p.scale * kLog2e;

  const bf16_t* qp = p.q + b * p.q_sb + h * p.q_sh;
  const int val = rw / (RW / 2);  // 0: this wave requests keys, 1: values
  const long long rst = val ? p.v_st : p.k_st;
  const u32x4 words = head_words(val ? p.v + b * p.v_sb + hk * p.v_sh : p.k + b * p.k_sb + hk * p.k_sh, rows_bytes(kv_end, rst, D));
  const Req req(rw % (RW / 2), lane, rst);
  char* const kbuf = smem + g * 2 * NB * TILE;
  char* const vbuf = kbuf + NB * TILE;
  char* const ring = val ? vbuf : kbuf;
  auto request = [&](int i, int place, int j) {  // (past the walk its last tile, which nobody reads)
    req(words, ring + place * TILE, __builtin_amdgcn_readfirstlane(key0(i) * (int)rst * 2), j);
  };
  auto requests = [&](int i, int place) {
#pragma unroll
    for (int j = 0; j < Req::N; ++j) request(i, place, j);
  };
  auto first = [&] {  // the places that the first step does not fill
#pragma unroll
    for (int i = 0; i < NB; ++i)
      if (i < NB - 1 || !val) requests(i, i);
  };
  first();
  bf16x8 qf[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s)
    qf[s] = *reinterpret_cast<const bf16x8*>(qp + (long long)min(qrow, p.Sq - 1) * p.q_st + 16 * s + 8 * hh);

  const int xr = (l32 >> 2) & 3;
  const int kb_e = (l32 >> 3) * 16 * D + 64 * (l32 & 7) + 16 * (hh ^ xr);
  const int kb_o = (l32 >> 3) * 16 * D + 64 * (l32 & 7) + 16 * ((2 + hh) ^ xr);
  const int c3 = 2 * ((lane >> 4) & 1) + ((gi & 3) >> 1);
  const int vb_1 = 64 * (4 * hh + (gi >> 2)) + 16 * (c3 ^ hh) + 8 * (gi & 1);
  const int vb_2 = 16 * D + 64 * (4 * hh + (gi >> 2)) + 16 * (c3 ^ hh ^ 2) + 8 * (gi & 1);
  auto qk = [&](const char* Ks, auto beside) {  // beside(s): after product s
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    bf16x8 fa[3];  // K fragments two k-steps ahead of their MFMA (pinned)
    fa[0] = lds_b128(Ks, kb_e);
    fa[1] = lds_b128(Ks, kb_o);
    __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      if (s + 2 < KS) {
        fa[(s + 2) % 3] = lds_b128(Ks, (((s + 2) & 1) ? kb_o : kb_e) + 512 * ((s + 2) >> 1));
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[s % 3], qf[s], acc, 0, 0, 0);
      __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
      beside(s);
    }
    return acc;
  };
  const int last = min(qrow + off, kv_end - 1);              // row's last visible key
  const int before = p.window > 0 ? qrow + off - p.window : -(1 << 30);            // key before its first
  auto mask = [&](f32x16& acc, int k0) {
    const int lim = last - k0 - 4 * hh, lo = before - k0 - 4 * hh;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int c = (r & 3) + 8 * (r >> 2);
      if (c > lim || c <= lo) acc[r] = -INFINITY;
    }
  };
  const float slope = G == 2 ? p.alibi[h] * kLog2e : 0.f;
  auto biased = [&](float s, int r, int k0) {  // score in log2 units
    return G == 2 ? fmaf(s, sl2, fmaf(slope, (float)((r & 3) + 8 * (r >> 2)), slope * (float)(k0 + 4 * hh - qrow - off))) : s * sl2;
  };

  if (tid == 0) again = 0;
  f32x16 oacc[D / 32];
  float m = -INFINITY, lsum = 0.f;
  bool begun = false;  // G == 1: a tile with a visible key of this row has been walked
  for (int pass = 0;; ++pass) {
    if (pass > 0) {  // a sum passed 2^100: the group's true maximum first
      m = -INFINITY;
      begun = true;
      for (int i = 0; i < nsteps; ++i) {
        if (!val) requests(i, 0);
        wait_and_meet<0>();
        f32x16 s = qk(kbuf, [](int) {});
        mask(s, mkey0(i));
#pragma unroll
        for (int r = 0; r < 16; ++r) m = fmaxf(m, s[r] == -INFINITY ? -INFINITY : biased(s[r], r, key0(i)));
        __syncthreads();
      }
      m = fmaxf(m, __shfl_xor(m, 32, 64));
      first();
    }
    clear<D>(oacc);
    lsum = 0.f;
    float nm = pass == 0 || m == -INFINITY ? 0.f : -m;
    wait_and_meet<(NB - 1) * Req::N>();
    f32x16 sa = qk(kbuf, [](int) {});

    auto step = [&](int i, f32x16& sa, f32x16& sb, auto masked) {
      constexpr bool MASKED = decltype(masked)::value, HEAD = decltype(masked)::value == 2;
      const int k0 = key0(i), mk0 = mkey0(i);
      // K(i + 1) and V(i) have landed, and all waves have read K(i) and V(i - 1): the next tiles go there
      wait_and_meet<(NB - 2) * Req::N>();
      sb = qk(kbuf + (i + 1) % NB * TILE, [&](int s) {  // S of the group's next tile (unused after the last)
        constexpr int EACH = KS / Req::N;
        static_assert(KS % Req::N == 0, "requests at even distances");
        if (s % EACH) return;
        __builtin_amdgcn_sched_barrier(0x406);
        request(i + NB - val, (i + NB - val) % NB, s / EACH);
        __builtin_amdgcn_sched_barrier(0x406);
      });
      float sl = sl2, bias[16];  // P = exp2(s * sl + bias)
      if constexpr (G == 2) {
        const float b0 = slope * (float)(k0 + 4 * hh - qrow - off) + (MASKED ? 0.f : nm);
#pragma unroll
        for (int r = 0; r < 16; ++r) bias[r] = fmaf(slope, (float)((r & 3) + 8 * (r >> 2)), b0);
      }
      if constexpr (MASKED) {
        mask(sa, mk0);
        float mt = -INFINITY, m_here = -INFINITY;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          sa[r] = G == 2 ? fmaf(sa[r], sl2, bias[r]) : sa[r] * sl2;
          mt = fmaxf(mt, sa[r]);
        }
        if constexpr (HEAD) {  // (the next tile's scores are at hand and may be the row's largest)
          m_here = fmaxf(mt, __shfl_xor(mt, 32, 64));
          const int nk0 = mkey0(i + 1), lim = last - nk0 - 4 * hh, lo = before - nk0 - 4 * hh;
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int c = (r & 3) + 8 * (r >> 2);
            mt = fmaxf(mt, c > lim || c <= lo ? -INFINITY : sb[r] * sl2);
          }
        }
        mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
        m = m == -INFINITY || (HEAD && !begun) ? mt : m;
        if constexpr (HEAD) begun = begun || m_here > -INFINITY;
        nm = m == -INFINITY ? 0.f : -m;
        sl = 1.f;
      }
      if constexpr (G < 2 || MASKED) {
#pragma unroll
        for (int r = 0; r < 16; ++r) bias[r] = nm;
      }
      float ps = 0.f;
      bf16x8 pf0, pf1;
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        const float e0 = __builtin_amdgcn_exp2f(fmaf(sa[r], sl, bias[r]));
        const float e1 = __builtin_amdgcn_exp2f(fmaf(sa[r + 8], sl, bias[r + 8]));
        ps += e0 + e1;
        pf0[r] = (__bf16)e0;
        pf1[r] = (__bf16)e1;
      }
      lsum += ps;
      const char* Vs = vbuf + i % NB * TILE;
      auto vfrag = [&](int db, int s) {
        return cat8(lds_tr4(Vs, vb_1 + 2 * s * 16 * D + 512 * db), lds_tr4(Vs, vb_2 + 2 * s * 16 * D + 512 * db));
      };
      bf16x8 va[2], vb[2];
      va[0] = vfrag(0, 0);
      vb[0] = vfrag(0, 1);
      __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
      for (int db = 0; db < D / 32; ++db) {
        if (db + 1 < D / 32) {
          va[(db + 1) & 1] = vfrag(db + 1, 0);
          vb[(db + 1) & 1] = vfrag(db + 1, 1);
          __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
        }
        oacc[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va[db & 1], pf0, oacc[db], 0, 0, 0);
        oacc[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vb[db & 1], pf1, oacc[db], 0, 0, 0);
        __builtin_amdgcn_sched_group_barrier(0x8, 2, 0);
      }
    };
    f32x16 sb;
    auto one = [&](int i, auto masked) {
      step(i, sa, sb, masked);
      sa = sb;
    };
    auto free = [&](int i, int end) {  // in pairs: no copy of the scores
      for (; i + 1 < end; i += 2) {
        step(i, sa, sb, std::false_type{});
        step(i + 1, sb, sa, std::false_type{});
      }
      if (i < end) one(i, std::false_type{});
    };
    if constexpr (G == 1) {
      // Steps whose KG tiles may hold a row's first visible key of their group: below f_lo the rows' first ones, up to
      // KG - 1 tiles on the other groups'. Free ones lie whole at or below f_hi.
      const int head = min(nsteps, (sp.f_lo - sp.lo + 2 * KG - 2) / KG);
      const int top = max(head, min(nsteps, (min(sp.f_hi + 1, sp.hi) - sp.lo) / KG));
      for (int i = 0; i < head; ++i) one(i, std::integral_constant<int, 2>{});
      free(head, top);
      for (int i = top; i < nsteps; ++i) one(i, std::true_type{});
    } else {
      // from the last tile down: a row's last visible key lies above f_hi, another group's up to KG - 1 tiles below
      const int top = min(nsteps, (sp.hi - 1 - sp.f_hi + 2 * KG - 2) / KG);
      const int low = max(top, min(sp.hi - sp.f_lo, ntiles) / KG);
      for (int i = 0; i < top; ++i) one(i, std::true_type{});
      free(top, low);
      for (int i = low; i < nsteps; ++i) one(i, std::true_type{});
    }

    // the groups' sums meet where the tiles were
    wait_and_meet<0>();
    const float ltot = lsum + __shfl_xor(lsum, 32, 64);
    const bool bad = !(ltot < 1.2676506e30f) && qrow < p.Sq;
    if (pass == 0 && __any(bad) && lane == 0) again = 1;
    if constexpr (KG > 1) {
      if (g > 0) put_partial<D>(smem + ((g - 1) * RW + rw) * PART, oacc, lane);
      if (hh == 0) {
        stat[g][rw][l32][0] = m;
        stat[g][rw][l32][1] = ltot;
      }
    }
    lsum = ltot;
    __syncthreads();
    if (pass > 0 || !__builtin_amdgcn_readfirstlane(again)) break;
  }
  if (KG > 1 && g > 0) return;
  float mm = m, l = lsum;
  if constexpr (KG > 1) {
#pragma unroll
    for (int i = 1; i < KG; ++i) mm = fmaxf(mm, stat[i][rw][l32][0]);
    auto weight = [&](float x) { return x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(x - mm); };
    const float w0 = weight(m);
    l *= w0;
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) oacc[db][r] *= w0;
#pragma unroll
    for (int i = 1; i < KG; ++i) {
      const float w = weight(stat[i][rw][l32][0]);
      l = fmaf(stat[i][rw][l32][1], w, l);
      add_partial<D>(smem + ((i - 1) * RW + rw) * PART, oacc, lane, w);
    }
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
  if (hh == 0 && p.lse && qrow < p.Sq) p.lse[((long long)b * p.H + h) * p.Sq + qrow] = l > 0.f ? (mm + log2f(l)) * kLn2 : INFINITY;
  asm volatile("" ::: "memory");  // (the image lies on the partial sums that this wave alone has read)
  store_tile_lds<D, D, true>(p.o + b * p.o_sb + h * p.o_sh + (long long)q0 * p.o_st, p.o_st, oacc, lane, inv, smem + rw * (KG > 1 ? PART : PART / 2),
                             p.Sq - q0);
}

// dQ: as the forward, a group walks every KG-th key tile of its 32 RW query rows; the groups' dQ add up in LDS.
template <int D, int G, int RW, int KG, int WPS>
__global__ void __launch_bounds__(64 * RW * KG, WPS) attn_bwd_dq_split_kernel(FastBwdParams p) {
  constexpr int BM = 32 * RW, BN = 32;
  constexpr int TILE = BN * D * 2, KS = D / 16;
  constexpr int NB = KG == 1 ? 4 : D == 128 ? 2 : 3;  // tiles of K and of V in LDS, a group
  using Req = TileRequests<D, RW / 2>;                // (half of a group's waves request K, the others V)
  constexpr int PART = 32 * D * 4;
  static_assert((KG - 1) * RW * PART <= KG * 2 * NB * TILE, "the partial sums take the tiles' place");
  __shared__ __attribute__((aligned(16))) char smem[KG * 2 * NB * TILE];  // per group [K's NB tiles | V's]

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = wave / RW, rw = wave % RW;
  const int l32 = lane & 31, hh = lane >> 5;
  const int nqb = (p.Sq + BM - 1) / BM, heads = p.B * p.H;
  const auto [qi, bh] = block_of<true, D, BM, WPS == 3 ? 3 : 1>(nqb, heads);
  const int qb = nqb - 1 - qi;
  const int b = bh / p.H, h = bh % p.H;
  const int hk = h / (p.H / p.Hkv);
  const int off = p.Sk - p.Sq;
  const int q0 = qb * BM + rw * 32, qrow = q0 + l32;
  const int kv_end = batch_keys(p.kv_len, b, p.Sk);
  const TileSpan sp = tile_span<BM, true>(qb * BM, off, kv_end, p.window);
  const int ntiles = sp.hi - sp.lo, nsteps = (ntiles + KG - 1) / KG;
  auto key0 = [&](int i) { return (sp.lo + min(KG * i + g, ntiles - 1)) * BN; };
  const float sl2 = p.scale * kLog2e;

  const int qr = min(qrow, p.Sq - 1);
  const bf16_t* qp = p.q + b * p.q_sb + h * p.q_sh + (long long)qr * p.q_st;
  const bf16_t* gp = p.dout + b * p.do_sb + h * p.do_sh + (long long)qr * p.do_st;
  const int val = rw / (RW / 2);  // 0: this wave requests keys, 1: values
  const long long rst = val ? p.v_st : p.k_st;
  const u32x4 words = head_words(val ? p.v + b * p.v_sb + hk * p.v_sh : p.k + b * p.k_sb + hk * p.k_sh, rows_bytes(kv_end, rst, D));
  const Req req(rw % (RW / 2), lane, rst);
  char* const kbuf = smem + g * 2 * NB * TILE;
  char* const vbuf = kbuf + NB * TILE;
  char* const ring = val ? vbuf : kbuf;
  auto request = [&](int i, int place, int j) { req(words, ring + place * TILE, __builtin_amdgcn_readfirstlane(key0(i) * (int)rst * 2), j); };
#pragma unroll
  for (int i = 0; i < NB - 1; ++i)
#pragma unroll
    for (int j = 0; j < Req::N; ++j) request(i, i, j);
  bf16x8 qf[KS], gf[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    qf[s] = *reinterpret_cast<const bf16x8*>(qp + 16 * s + 8 * hh);
    gf[s] = *reinterpret_cast<const bf16x8*>(gp + 16 * s + 8 * hh);
  }
  const float slope = G == 2 ? p.alibi[h] * kLog2e : 0.f;
  const long long li = ((long long)b * p.H + h) * p.Sq + qr;
  const float nlse = -p.lse[li] * kLog2e;
  float dl = 0.f;  // delta = rowsum(dO * O), left for the dK/dV kernel too
  {
    const bf16_t* op = p.o + b * p.o_sb + h * p.o_sh + (long long)qr * p.o_st;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const bf16x8 of = *reinterpret_cast<const bf16x8*>(op + 16 * s + 8 * hh);
#pragma unroll
      for (int j = 0; j < 8; ++j) dl = fmaf((float)of[j], (float)gf[s][j], dl);
    }
    dl += __shfl_xor(dl, 32, 64);
    if (g == 0 && hh == 0 && qrow < p.Sq) p.delta[li] = dl;
  }
  f32x16 dq[D / 32];
  clear<D>(dq);
  int be, bo, b1, b2;
  row_bases<D>(l32, hh, be, bo);
  tr_bases<D>(lane, b1, b2);
  const int last = min(qrow + off, kv_end - 1);    // row's last visible key
  const int before = p.window > 0 ? qrow + off - p.window : -(1 << 30);  // key before its first

  auto step = [&](int i, auto masked) {
    constexpr bool MASKED = decltype(masked)::value;
    const int k0 = key0(i);
    const char* Ks = kbuf + i % NB * TILE;
    const char* Vs = vbuf + i % NB * TILE;
    // tile i has landed, and all waves have read tile i - 1: the next one goes there
    wait_and_meet<(NB - 2) * Req::N>();
    f32x16 st, dpt;
#pragma unroll
    for (int r = 0; r < 16; ++r) { st[r] = 0.f; dpt[r] = 0.f; }
    {  // K / V row fragments two k-steps ahead of their MFMAs (pinned)
      bf16x8 fk[3], fv[3];
      fk[0] = row_frag<D>(Ks, be, bo, 0);
      fv[0] = row_frag<D>(Vs, be, bo, 0);
      fk[1] = row_frag<D>(Ks, be, bo, 1);
      fv[1] = row_frag<D>(Vs, be, bo, 1);
      __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        if (s + 2 < KS) {
          fk[(s + 2) % 3] = row_frag<D>(Ks, be, bo, s + 2);
          fv[(s + 2) % 3] = row_frag<D>(Vs, be, bo, s + 2);
          __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        }
        st = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fk[s % 3], qf[s], st, 0, 0, 0);
        dpt = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fv[s % 3], gf[s], dpt, 0, 0, 0);
        __builtin_amdgcn_sched_group_barrier(0x8, 2, 0);
        constexpr int EACH = KS / Req::N;
        static_assert(KS % Req::N == 0, "requests at even distances");
        if (s % EACH == 0) {  // (all waves' at once hold the products up)
          __builtin_amdgcn_sched_barrier(0x406);
          request(i + NB - 1, (i + NB - 1) % NB, s / EACH);
          __builtin_amdgcn_sched_barrier(0x406);
        }
      }
    }
    // visible key offsets (r&3)+8(r>>2): lo < offset <= lim
    const int mk0 = KG * i + g < ntiles ? k0 : kNoTile;
    const int lim = last - mk0 - 4 * hh, lo = before - mk0 - 4 * hh;
    const float b0 = G == 2 ? fmaf(slope, (float)(k0 + 4 * hh - qrow - off), nlse) : nlse;
    bf16x8 d0, d1;
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const int c = (r & 3) + 8 * (r >> 2);
      float p0 = __builtin_amdgcn_exp2f(fmaf(st[r], sl2, G == 2 ? fmaf(slope, (float)c, b0) : b0));
      float p1 = __builtin_amdgcn_exp2f(fmaf(st[r + 8], sl2, G == 2 ? fmaf(slope, (float)(c + 16), b0) : b0));
      if constexpr (MASKED) {
        if (c > lim || c <= lo) p0 = 0.f;
        if (c + 16 > lim || c + 16 <= lo) p1 = 0.f;
      }
      d0[r] = (__bf16)(p0 * (dpt[r] - dl));
      d1[r] = (__bf16)(p1 * (dpt[r + 8] - dl));
    }
    {
      bf16x8 t0[2], t1[2];
      t0[0] = tr_frag<D>(Ks, b1, b2, 0, 0);
      t1[0] = tr_frag<D>(Ks, b1, b2, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
      for (int db = 0; db < D / 32; ++db) {
        if (db + 1 < D / 32) {
          t0[(db + 1) & 1] = tr_frag<D>(Ks, b1, b2, 0, db + 1);
          t1[(db + 1) & 1] = tr_frag<D>(Ks, b1, b2, 1, db + 1);
          __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
        }
        dq[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(t0[db & 1], d0, dq[db], 0, 0, 0);
        dq[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(t1[db & 1], d1, dq[db], 0, 0, 0);
        __builtin_amdgcn_sched_group_barrier(0x8, 2, 0);
      }
    }
  };
  const int low = min(nsteps, (max(0, sp.f_lo - sp.lo) + KG - 1) / KG);
  const int top = max(low, min(nsteps, (min(sp.f_hi + 1, sp.hi) - sp.lo) / KG));
  for (int i = 0; i < low; ++i) step(i, std::true_type{});
  for (int i = low; i < top; ++i) step(i, std::false_type{});
  for (int i = top; i < nsteps; ++i) step(i, std::true_type{});

  wait_and_meet<0>();  // what comes next lies where the tiles were
  if constexpr (KG > 1) {
    if (g > 0) put_partial<D>(smem + ((g - 1) * RW + rw) * PART, dq, lane);
    __syncthreads();
    if (g > 0) return;
#pragma unroll
    for (int i = 1; i < KG; ++i) add_partial<D>(smem + ((i - 1) * RW + rw) * PART, dq, lane, 1.f);
    asm volatile("" ::: "memory");
  }
  store_tile_lds<D, D, true>(p.dq + b * p.dq_sb + h * p.dq_sh + (long long)q0 * p.dq_st, p.dq_st, dq, lane, p.scale,
                             smem + rw * (KG > 1 ? PART : PART / 2), p.Sq - q0);
}

// dK/dV: a wave has 32 keys of the workgroup's 32 RW and its group every KG-th 32-row tile of Q and dO (of all the query heads
// of a KV head); the groups' dV, then their dK add up in LDS.
template <int D, int G, bool WIN, int RW, int KG, int WPS>
__global__ void __launch_bounds__(64 * RW * KG, WPS) attn_bwd_dkdv_split_kernel(FastBwdParams p) {
  constexpr int BK = 32 * RW, BQ = 32, NTG = 64 * RW;
  // The sums start with a row's -lse (over the scale) and -delta: no LDS read is left to wait for behind the products, where no register
  // is free to hold them, and the subtractions go. dK/dV, us: 64 wide, one group, 8 x 1000 x 12 heads 47.2 -> 41.3, 6 x 1024 x 16 46.8 ->
  // 42.4, 16 x 380 x 12 21.3 -> 19.6; 128 wide, two groups, 2048 x 14 with ALiBi 75.9 -> 72.2, 700 x 20 25.0 -> 24.3. ALiBi and windows
  // spill at 64 (51.9 -> 61.2), 64 wide in two groups, 96 wide and 128 wide in one gain and lose 4 %.
  constexpr bool START = D == 64 ? KG == 1 && G == 1 && !WIN : D == 128 && KG == 2;
  constexpr int TILE = BQ * D * 2, KS = D / 16, NCH = D / 8;
  using Req = TileRequests<D, RW / 2>;  // (half of a group's waves request Q, the others dO)
  constexpr int PART = 32 * D * 4;
  static_assert((KG - 1) * RW * PART <= KG * 4 * TILE, "the partial sums take the tiles' place");
  constexpr int VOFF = KG * 4 * TILE;  // V images of the RW key blocks, the groups' alike
  constexpr int LOFF = VOFF + RW * TILE;
  __shared__ __attribute__((aligned(16))) char smem[LOFF + KG * 2 * 64 * 4];  // lse / delta: [group][buf][64] floats

  const int tid = threadIdx.x, lane = tid & 63, gt = tid % NTG;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = wave / RW, rw = wave % RW;
  const int l32 = lane & 31, hh = lane >> 5;
  const int heads = p.B * p.Hkv;
  const auto [kb, bh] = block_of<true, D, BK, D == 64 ? 3 : 1>((p.Sk + BK - 1) / BK, heads);
  const int b = bh / p.Hkv, hk = bh % p.Hkv;
  const int grp = p.H / p.Hkv;
  const int off = p.Sk - p.Sq;
  const int kw = kb * BK + rw * 32, key = kw + l32;
  const int kv_end = batch_keys(p.kv_len, b, p.Sk);
  const float sl2 = p.scale * kLog2e, inv = 1.f / p.scale;

  const int q_lo = max(0, kb * BK - off) & ~(BQ - 1);
  // no query sees a block past the length; past the last key's window no query sees the block
  const int q_end = WIN ? min(p.Sq, kb * BK + BK - 1 - off + p.window) : p.Sq;
  const int nqt = max(0, q_end - q_lo + BQ - 1) / BQ;
  const int total = kb * BK < kv_end ? nqt * grp : 0, nsteps = (total + KG - 1) / KG;
  const int grad = rw / (RW / 2);  // 0: this wave requests queries, 1: output gradients
  const long long rst = grad ? p.do_st : p.q_st, rsh = grad ? p.do_sh : p.q_sh;
  const bf16_t* const rbase = grad ? p.dout + b * p.do_sb : p.q + b * p.q_sb;
  const int rbytes = rows_bytes(p.Sq, rst, D);
  const Req req(rw % (RW / 2), lane, rst);
  char* const own = smem + g * 4 * TILE;
  float* const stat = reinterpret_cast<float*>(smem + LOFF) + g * 128;
  char* const ring = own + grad * TILE;
  float lreg = 0.f;
  int be, bo, b1, b2;
  row_bases<D>(l32, hh, be, bo);
  tr_bases<D>(lane, b1, b2);

  // The group's current tile: query head hcur of the KV head, q tile qcur; past its last one the tile stays and is masked.
  int hcur = 0, qcur = 0, tile = g;
  auto settle = [&] {  // (after qcur moved on)
    while (qcur >= nqt && hcur < grp - 1) qcur -= nqt, ++hcur;
    qcur = min(qcur, nqt - 1);
  };
  auto tile_words = [&] { return head_words(rbase + (hk * grp + hcur) * rsh, rbytes); };
  auto request = [&](const u32x4& words, int buf, int j) {
    req(words, ring + buf * 2 * TILE, __builtin_amdgcn_readfirstlane((q_lo + qcur * BQ) * (int)rst * 2), j);
  };
  auto load_stat = [&] {
    if (gt < 64) {  // as they come: the scaling waits until they are stored
      const long long li = ((long long)b * p.H + hk * grp + hcur) * p.Sq + min(q_lo + qcur * BQ + (gt & 31), p.Sq - 1);
      lreg = (gt < 32 ? p.lse : p.delta)[li];
    }
  };
  auto store_stat = [&](int buf) {
    if (gt < 64) {
      float v = lreg;
      if (q_lo + qcur * BQ + (gt & 31) >= p.Sq) v = gt < 32 ? INFINITY : 0.f;  // P = 0
      stat[buf * 64 + gt] = !START ? (gt < 32 ? v * kLog2e : v) : gt < 32 ? -v * inv : -v;
    }
  };
  if (total > 0) {  // (flies with the key and value rows)
    qcur = g;
    settle();
    const u32x4 words = tile_words();
#pragma unroll
    for (int j = 0; j < Req::N; ++j) request(words, 0, j);
    load_stat();
  }
  const bf16_t* kp = p.k + b * p.k_sb + hk * p.k_sh;
  const bf16_t* vp = p.v + b * p.v_sb + hk * p.v_sh;
  bf16x8 kf[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    kf[s] = *reinterpret_cast<const bf16x8*>(kp + (long long)min(key, p.Sk - 1) * p.k_st + 16 * s + 8 * hh);
    if (key >= kv_end) kf[s] = bf16x8{};
  }
  // V rows -> the images (read back by rows for dP), 32 RW rows over all threads
  constexpr int NT = NTG * KG;
  char* const vimg = smem + VOFF + rw * TILE;
#pragma unroll
  for (int i = 0; i < (BK * NCH + NT - 1) / NT; ++i) {
    const int idx = tid + NT * i, row = idx / NCH, ch = idx % NCH;
    if (BK * NCH % NT == 0 || idx < BK * NCH) {
      const u32x4 x = *reinterpret_cast<const u32x4*>(vp + (long long)min(kb * BK + row, p.Sk - 1) * p.v_st + ch * 8);
      *reinterpret_cast<u32x4*>(smem + VOFF + (row / 32) * TILE + img_off<D>(row % 32, ch)) =
          kb * BK + row < kv_end ? x : u32x4{0, 0, 0, 0};
    }
  }
  f32x16 dk[D / 32], dv[D / 32];
  clear<D>(dk);
  clear<D>(dv);

  if (total > 0) store_stat(0);
  wait_and_meet<0>();
  for (int i = 0; i < nsteps; ++i) {
    const int qt = q_lo + qcur * BQ, hq = hk * grp + hcur;
    const bool gone = tile >= total;
    // Tiles below the diagonal and inside the window skip the mask. (D = 64 has no registers for two ways through the softmax at
    // 3 waves a SIMD; two bodies of the whole step spill at every D. 1 x 1500 x 64 heads of 96: 150 -> 142 us with dQ.)
    const bool plain = D > 64 && !gone && kb * BK + BK <= kv_end && kb * BK + BK - 1 <= qt + off &&
                       (!WIN || kb * BK > qt + BQ - 1 + off - p.window);
    const char* Qs = own + (i & 1) * 2 * TILE;
    const char* Gs = Qs + TILE;
    const float* ls = stat + (i & 1) * 64;
    tile += KG;
    qcur += KG;
    settle();
    load_stat();
    const u32x4 words = tile_words();
    asm volatile("" ::: "memory");
    f32x16 sacc, dpacc;
#pragma unroll
    for (int gg = 0; gg < 4; ++gg) {
      if constexpr (!START) {
#pragma unroll
        for (int j = 0; j < 4; ++j) sacc[4 * gg + j] = dpacc[4 * gg + j] = 0.f;
        continue;
      }
      const f32x4 lq = *reinterpret_cast<const f32x4*>(ls + 8 * gg + 4 * hh), dq4 = *reinterpret_cast<const f32x4*>(ls + 32 + 8 * gg + 4 * hh);
#pragma unroll
      for (int j = 0; j < 4; ++j) sacc[4 * gg + j] = lq[j], dpacc[4 * gg + j] = dq4[j];
    }
    if constexpr (START) __builtin_amdgcn_sched_barrier(0);
    {  // S = Q.K^T, dP = dO.V^T, the three fragments of k-step s + 1 before the MFMAs of step s (pinned)
      bf16x8 fq[2], fg[2], fv[2];
      fq[0] = row_frag<D>(Qs, be, bo, 0), fg[0] = row_frag<D>(Gs, be, bo, 0), fv[0] = row_frag<D>(vimg, be, bo, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        if (s + 1 < KS) {
          fq[(s + 1) & 1] = row_frag<D>(Qs, be, bo, s + 1);
          fg[(s + 1) & 1] = row_frag<D>(Gs, be, bo, s + 1);
          fv[(s + 1) & 1] = row_frag<D>(vimg, be, bo, s + 1);
          __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
        }
        sacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fq[s & 1], kf[s], sacc, 0, 0, 0);
        dpacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fg[s & 1], fv[s & 1], dpacc, 0, 0, 0);
        __builtin_amdgcn_sched_group_barrier(0x8, 2, 0);
        constexpr int EACH = KS / Req::N;
        static_assert(KS % Req::N == 0, "requests at even distances");
        if (s % EACH == 0) {  // the next tile, where all waves have read the one before (all waves' requests at once hold the products up)
          __builtin_amdgcn_sched_barrier(0x406);
          request(words, (i + 1) & 1, s / EACH);
          __builtin_amdgcn_sched_barrier(0x406);
        }
      }
    }
    // rows q = qt + 8g + 4hh + j (g = r>>2, j = r&3) that see the key: lim <= 8g + j < ul
    int lim = key - qt - off - 4 * hh;
    if (key >= kv_end || gone) lim = 1 << 30;
    const int ul = WIN ? key + p.window - off - qt - 4 * hh : 0;
    float slope = 0.f, b0 = 0.f;
    if constexpr (G == 2) {
      slope = p.alibi[hq] * kLog2e;
      b0 = slope * (float)(key - qt - off - 4 * hh);
    }
    float pr[16];
#pragma unroll
    for (int gg = 0; gg < 4; ++gg) {
      f32x4 lq{0.f, 0.f, 0.f, 0.f};
      if constexpr (!START) lq = *reinterpret_cast<const f32x4*>(ls + 8 * gg + 4 * hh);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float bl = G == 2 ? fmaf(-slope, (float)(8 * gg + j), b0) - lq[j] : -lq[j];
        pr[4 * gg + j] = __builtin_amdgcn_exp2f(START && G != 2 ? sacc[4 * gg + j] * sl2 : fmaf(sacc[4 * gg + j], sl2, bl));
      }
    }
    if (!plain) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int c = 8 * (r >> 2) + (r & 3);
        if (c < lim || (WIN && c >= ul)) pr[r] = 0.f;
      }
    }
    bf16x8 p0, p1, s0, s1;
#pragma unroll
    for (int gg = 0; gg < 4; ++gg) {
      f32x4 dq4{0.f, 0.f, 0.f, 0.f};
      if constexpr (!START) dq4 = *reinterpret_cast<const f32x4*>(ls + 32 + 8 * gg + 4 * hh);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int r = 4 * gg + j;
        const float ds = pr[r] * (START ? dpacc[r] : dpacc[r] - dq4[j]);
        if (r < 8) { p0[r] = (__bf16)pr[r]; s0[r] = (__bf16)ds; }
        else { p1[r - 8] = (__bf16)pr[r]; s1[r - 8] = (__bf16)ds; }
      }
    }
    {  // dV^T += dO^T.P, dK^T += Q^T.dS: the reads of d-block db + 1 under the MFMAs of block db (pinned)
      bf16x8 fr[2][4];
      auto get = [&](int db) {
        fr[db & 1][0] = tr_frag<D>(Gs, b1, b2, 0, db), fr[db & 1][1] = tr_frag<D>(Gs, b1, b2, 1, db);
        fr[db & 1][2] = tr_frag<D>(Qs, b1, b2, 0, db), fr[db & 1][3] = tr_frag<D>(Qs, b1, b2, 1, db);
        __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);
      };
      get(0);
#pragma unroll
      for (int db = 0; db < D / 32; ++db) {
        if (db + 1 < D / 32) get(db + 1);
        dv[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[db & 1][0], p0, dv[db], 0, 0, 0);
        dv[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[db & 1][1], p1, dv[db], 0, 0, 0);
        dk[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[db & 1][2], s0, dk[db], 0, 0, 0);
        dk[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[db & 1][3], s1, dk[db], 0, 0, 0);
        __builtin_amdgcn_sched_group_barrier(0x8, 4, 0);
      }
    }
    asm volatile("" ::: "memory");
    if (i + 1 < nsteps) store_stat((i + 1) & 1);
    wait_and_meet<0>();
  }
  // group 0 adds dV up and stores it, then the last group dK
  if constexpr (KG > 1) {
    if (g > 0) put_partial<D>(smem + ((g - 1) * RW + rw) * PART, dv, lane);
    __syncthreads();
    if (g == 0) {
#pragma unroll
      for (int i = 1; i < KG; ++i) add_partial<D>(smem + ((i - 1) * RW + rw) * PART, dv, lane, 1.f);
    }
    __syncthreads();
    if (g < KG - 1) put_partial<D>(smem + (g * RW + rw) * PART, dk, lane);
    __syncthreads();
    if (g == KG - 1) {
#pragma unroll
      for (int i = 0; i < KG - 1; ++i) add_partial<D>(smem + (i * RW + rw) * PART, dk, lane, 1.f);
    }
    asm volatile("" ::: "memory");
  }
  if (KG > 1 && g > 0 && g < KG - 1) return;
  // (images of this wave's own: KG = 1, in the tiles; else group 0's in the V images, the last group's on what it has read)
  char* const img = KG == 1 ? smem + rw * (PART / 2) : g == 0 ? vimg : smem + rw * PART;
  if (g == 0)
    store_tile_lds<D, D, true>(p.dv + b * p.dv_sb + hk * p.dv_sh + (long long)kw * p.dv_st, p.dv_st, dv, lane, 1.f, img, p.Sk - kw);
  if (g == KG - 1)
    store_tile_lds<D, D, true>(p.dk + b * p.dk_sb + hk * p.dk_sh + (long long)kw * p.dk_st, p.dk_st, dk, lane, p.scale, img, p.Sk - kw);
}

}  // namespace

// Which calls are split in two groups (two waves of 32 rows each, 4 waves a workgroup) and which take blocks of 128 rows and one group.
// A split costs each of its blocks the meeting of the sums, so it wins as long as all of its blocks of 64 rows run at one time (three
// workgroups a CU of 64-wide heads, 768 in all, two of others, 512); with walks of up to three tiles only while they are one a CU. Past
// that, a causal call's longest blocks stand alone at the end, the more the longer they are, and a split halves them: the line rises with the
// longest walk (keys that a row sees; dK/dV: queries). dK/dV in two groups has short tiles to itself and gains further out. One MI355X, random
// calls of 24 to 5400 rows (none, ALiBi, lengths, windows), 12 000 in all: the form that these lines pick is 0.03 to 0.3 % slower than the
// better of the two on average. us with one group and with two at so many blocks of 64 rows:
//   forward, 64 wide:  128 rows, 640 10.2, 9.5; 784 11.7, 14.2; 512 rows, 768 12.9, 12.0; 784 13.4, 14.6; 600 rows, 780 14.4, 16.4; 1280 rows, 800 22.0, 19.2; 1280, 1080 24.5, 25.2; 2304, 1152 42, 40; 1296 47, 47
//   96 wide:           192 rows, 252 (168 of 128 rows) 8.8, 8.5; 264 (176) 9.0, 9.7; 396 (264) 11.4, 10.7; 512 rows, 440 14.3, 13.0; 520 14.6, 16.0; 1024, 512 20.6, 17.6; 608 21.4, 22.0; 2048, 720 43, 41
//   128 wide:          256 rows, 280 12.2, 11.5; 512, 512 18.6, 16.4; 640 21, 24; 1111, 504 27, 23; 1152, 648 27.2, 26.3; 1280, 720 30, 33; 1838, 638 42, 36
// Windows: a block of 128 rows sees as many keys more. All their blocks have as much to do, so none stands alone at the end. (With the
// window alone as the walk, 4 x 320 rows of 12 heads of 64 with a window of 69 took 10.8 us in one group; two take 8.0.)
struct Upto { int walk, blocks; };
template <int N>
static int blocks_upto(const Upto (&t)[N], int walk) {
  int b = -1;
  for (const Upto& u : t)
    if (walk >= u.walk) b = u.blocks;
  return b;
}
static int longest_walk(int rows, int window) { return window > 0 && window < rows ? min(rows, min(window + 128, 512)) : rows; }
static long long halves(int rows, int heads) { return (rows + 63ll) / 64 * heads; }
static bool split_rows(int rows, int heads, int d, int keys, int window, bool dq) {
  static const Upto f64[] = {{33, 260}, {97, 768}, {850, 790}, {1000, 880}, {1900, 1200}}, q64[] = {{65, 260}, {256, 768}, {900, 1000}, {1400, 1200}};
  static const Upto f96[] = {{65, 270}, {129, 520}, {900, 600}, {1400, 640}, {1900, 740}, {3000, 840}};
  static const Upto q96[] = {{65, 260}, {256, 512}, {700, 640}, {1000, 800}, {2300, 950}};
  static const Upto f128[] = {{33, 258}, {129, 514}, {1000, 640}, {1400, 720}, {2300, 800}, {3500, 900}};
  static const Upto q128[] = {{65, 260}, {256, 500}, {700, 600}, {1000, 800}, {2300, 1000}};
  const int walk = longest_walk(keys, window);
  const int upto = d == 64   ? (dq ? blocks_upto(q64, walk) : blocks_upto(f64, walk))
                   : d == 96 ? (dq ? blocks_upto(q96, walk) : blocks_upto(f96, walk))
                             : (dq ? blocks_upto(q128, walk) : blocks_upto(f128, walk));
  // Two blocks of few tiles a head, forward: one group, too, while its blocks are one a CU and those of 64 rows would be two. (Not windows, whose
  // blocks have less to do each: 8 x 300 rows of 8 heads of 96, a window of 16 to 90, two take .80 to .89 of one's time.)
  const long long blocks = (rows + 127ll) / 128 * heads;
  if (d != 64 && !dq && keys > 128 && keys <= 220 && blocks > 170 && blocks <= 256 && !(window > 0 && window < keys)) return false;
  return halves(rows, heads) <= upto;
}
// dK/dV with one group or two, or, 128 wide, 0, 1 or in two groups of four waves (2, by blocks of 128 rows): there two groups of two take 81 KB of
// LDS, one workgroup a CU. us, backward with one group, and what two groups (of four waves) take or save:
//   64 wide:   200 rows, 680 blocks of 64 rows 22.9, -0.7; 800 23.3, +1.1; 768, 600 43.5, +1.0; 1200, 912 61.3, -2.9; 3500, 1320 170, -5.2; 1485 188, +5.3
//   96 wide:   64 rows, 1200 50.2, -3.9; 200, 440 25.0, -0.6; 520 28.7, +1.5; 768, 684 52.8, -0.8; 804 55.7, +2.1; 1500, 960 96.8, -1.9; 1128 110, +8
//   128 wide:  200 rows, 200 26.0, -1.9 (-1.0); 512, 280 43.1, -4.8 (-4.1); 360 44.0, -0.9 (-3.8); 520 48.9, +7.8 (-2.2); 600 51.0, +9.7 (+0.6); 1024, 672 77.9,
//              +8.5 (-6.6); 2048, 448 117, -16 (-17); 1120 170, +35 (-2.0); 1280 172, +43 (+1.7); 4096, 512 226, -40 (-37); 1280 315, +54 (-7)
static int split_keys(int keys, int heads, int d, int rows, int window) {
  static const Upto t64[] = {{33, 1 << 30}, {65, 770}, {400, 970}, {900, 1400}}, t96[] = {{0, 1 << 30}, {65, 516}, {400, 700}, {700, 860}, {1700, 1100}};
  static const Upto t128[] = {{33, 258}, {700, 340}, {1200, 384}, {1700, 416}, {2600, 450}}, w128[] = {{97, 260}, {640, 553}};
  const int walk = longest_walk(rows, window);
  if (halves(keys, heads) <= (d == 64 ? blocks_upto(t64, walk) : d == 96 ? blocks_upto(t96, walk) : blocks_upto(t128, walk))) return 1;
  return d == 128 && (keys + 127ll) / 128 * heads <= blocks_upto(w128, walk) ? 2 : 0;
}

template <class F>
static int with_form(int d, bool alibi, F&& f) {
  auto mask = [&](auto D) {
    if (alibi) f(D, std::integral_constant<int, 2>{});
    else f(D, std::integral_constant<int, 1>{});
  };
  switch (d) {
    case 64: mask(std::integral_constant<int, 64>{}); break;
    case 96: mask(std::integral_constant<int, 96>{}); break;
    case 128: mask(std::integral_constant<int, 128>{}); break;
    default: return 1;
  }
  return hipGetLastError() == hipSuccess ? 0 : 3;
}

// Causal calls of 64, 96 and 128 wide heads with 16-byte rows; 1: another head size (or, backward, a scale of nothing).
// 96-wide rows in one group: three workgroups a CU where there are more than two, though their registers are then tight (1 x 1500 x 64 forward 53
// -> 46 us, backward 139 -> 134; up to 512 blocks of 128 rows the third never runs, and the forward takes 1 to 2 % longer, the whole
// backward 2 to 3 %). ALiBi's dQ would spill.
int attn_fwd_split(const FastFwdParams& p, int d, hipStream_t stream) {
  const long long blocks = (long long)((p.Sq + 127) / 128) * p.B * p.H;
  const bool two = split_rows(p.Sq, p.B * p.H, d, p.Sk, p.window, false);
  return with_form(d, p.alibi, [&](auto D_, auto G_) {
    constexpr int D = decltype(D_)::value, G = decltype(G_)::value, W = D == 64 ? 3 : 2;
    if (two)
      hipLaunchKernelGGL((attn_fwd_split_kernel<D, G, 2, 2, W>), dim3((p.Sq + 63) / 64 * p.B * p.H), dim3(256), 0, stream, p);
    else if (D == 96 && blocks > 512)
      hipLaunchKernelGGL((attn_fwd_split_kernel<D, G, 4, 1, D == 96 ? 3 : W>), dim3((unsigned)blocks), dim3(256), 0, stream, p);
    else
      hipLaunchKernelGGL((attn_fwd_split_kernel<D, G, 4, 1, W>), dim3((unsigned)blocks), dim3(256), 0, stream, p);
  });
}

int attn_bwd_split(const FastBwdParams& p, int d, hipStream_t stream) {
  if (!(fabsf(p.scale) >= 1e-30f)) return 1;  // the sums start with lse / scale: the generic kernel's
  const long long qblocks = (long long)((p.Sq + 127) / 128) * p.B * p.H, kblocks = (long long)((p.Sk + 127) / 128) * p.B * p.Hkv;
  const bool two = split_rows(p.Sq, p.B * p.H, d, p.Sk, p.window, true);
  const int kv = split_keys(p.Sk, p.B * p.Hkv, d, p.Sq, p.window);
  return with_form(d, p.alibi, [&](auto D_, auto G_) {
    constexpr int D = decltype(D_)::value, G = decltype(G_)::value, W = D == 64 ? 3 : 2;
    if (two)
      hipLaunchKernelGGL((attn_bwd_dq_split_kernel<D, G, 2, 2, W>), dim3((p.Sq + 63) / 64 * p.B * p.H), dim3(256), 0, stream, p);
    else if (D == 96 && G == 1 && qblocks > 512)
      hipLaunchKernelGGL((attn_bwd_dq_split_kernel<D, G, 4, 1, D == 96 && G == 1 ? 3 : W>), dim3((unsigned)qblocks), dim3(256), 0, stream, p);
    else
      hipLaunchKernelGGL((attn_bwd_dq_split_kernel<D, G, 4, 1, W>), dim3((unsigned)qblocks), dim3(256), 0, stream, p);
    auto dkdv = [&](auto WIN_) {
      constexpr bool WIN = decltype(WIN_)::value;
      if (kv == 1)
        hipLaunchKernelGGL((attn_bwd_dkdv_split_kernel<D, G, WIN, 2, 2, W>), dim3((p.Sk + 63) / 64 * p.B * p.Hkv), dim3(256), 0,
                           stream, p);
      else if (kv == 0)
        hipLaunchKernelGGL((attn_bwd_dkdv_split_kernel<D, G, WIN, 4, 1, W>), dim3((unsigned)kblocks), dim3(256), 0, stream, p);
      if constexpr (D == 128)
        if (kv == 2)
          hipLaunchKernelGGL((attn_bwd_dkdv_split_kernel<D, G, WIN, 4, 2, 2>), dim3((unsigned)kblocks), dim3(512), 0, stream, p);
    };
    if (p.window > 0) dkdv(std::true_type{});
    else dkdv(std::false_type{});
  });
}
