// Flash attention, backward of 256-wide heads: a pair of waves shares what one wave's registers held.
//
// What bounds these calls. A wave of attn_bwd_dkdv_tiled_kernel holds dK and dV of its 32 keys: half of a SIMD's registers, with K's
// fragments, the tile's loads and the products' operands nearly all of them, so that a SIMD runs one wave whose products, softmax,
// LDS reads and barriers follow each other (5000 cycles a tile, 2048 of them in the matrix cores). dQ's wave, with Q, dO and dQ, is no
// smaller. Here the 32 keys (rows) are a pair of waves' and a SIMD runs two.
//   dK/dV: the first takes S = Q.K^T, P and dV^T += dO^T.P, the second dP = dO.V^T, dS and dK^T += Q^T.dS, each with 128 accumulator
//          registers and the 64 of its K or V rows. V's rows are no longer read from LDS (a fifth of its reads).
//   dQ:    the first takes S^T = K.Q^T and P, the second dP^T = V.dO^T, dS^T and dQ^T += K^T.dS^T, and leaves delta = rowsum(dO * O).
// P goes from one to the other through LDS, in fp32 as it was. The second wave runs a tile behind and turns its step around -- dS and
// its last product of tile t - 1, then dP of tile t -- so that one's softmax lies beside the other's products, and leaves the loads to the
// first one, which has less to do: requests straight into LDS (TileRequests), two steps ahead, one between two products.
//
// Backward, us, one wave and a pair: 2 x 2048 x 16 heads 300, 266; 1 x 2048 225, 184; 1 x 4096 522, 454; 4 x 1100 234, 198; 8 x 512
// with lengths 128, 108; 1 x 3000 with ALiBi 361, 285; 3 x 300 56, 46; 1 x 61 24.7, 21.8. That was with tiles through the first wave's registers,
// for which the last quarter of K's fragments had to lie in LDS and be read again at each step; requested into LDS, pairs, before and now:
// 2 x 2048 254, 241 (dK/dV 137, 129; dQ 114, 108); 1 x 2048 182, 166; 1 x 4096 447, 420; 1 x 3000 with ALiBi 278, 259; 3 x 300 46.7, 44.1.
// What bounds them: the LDS reads of both waves, 256 KB of a step of dK/dV, 192 of dQ (2048, 1536 cycles at 128 bytes), beside as many cycles in
// the matrix cores, and what of a wave's own chain the other does not cover. No gain: deeper rings of fragments, wave priorities, a walk that touches
// tiles ahead, heads turned over the XCDs, dQ's columns half to the first wave, with dS through LDS (130, 137: the reads stay as many).
#include "attn_fast.h"

#include <type_traits>

namespace {

struct Nothing { __device__ void operator()(int) const {} };

// Rows of a tile image times a fixed operand, the reads two steps ahead of their product (pinned), `also(s)` between
template <int D, class Also = Nothing>
__device__ __forceinline__ f32x16 pair_rows(const char* smem, int img, int be, const bf16x8 (&fix)[D / 16], Also also = {}) {
  constexpr int KS = D / 16;
  f32x16 x;
#pragma unroll
  for (int r = 0; r < 16; ++r) x[r] = 0.f;
  bf16x8 f[3];
  const int e = be + img, o = e ^ 32;  // (row_bases' second one is made of the first: the registers are full)
  __builtin_amdgcn_sched_barrier(0);  // (earlier reads are not of the groups)
  f[0] = row_frag<D>(smem, e, o, 0), f[1] = row_frag<D>(smem, e, o, 1);
  __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const int t = s + 2;
    if (t < KS) {
      f[t % 3] = row_frag<D>(smem, e, o, t);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    also(s);
    x = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[s % 3], fix[s], x, 0, 0, 0);
    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
  }
  return x;
}

// acc += a tile image's columns times (x0, x1), read like its rows
template <int D>
__device__ __forceinline__ void pair_columns(f32x16 (&acc)[D / 32], const char* smem, int img, int b1, bf16x8 x0, bf16x8 x1) {
  bf16x8 f[3];
  const int c1 = b1 + img, c2 = (c1 ^ 32) + 16 * D;
  auto get = [&](int n) {
    f[n % 3] = tr_frag<D>(smem, c1, c2, n & 1, n >> 1);
    __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
  };
  __builtin_amdgcn_sched_barrier(0);
  get(0);
  get(1);
#pragma unroll
  for (int n = 0; n < D / 16; ++n) {
    if (n + 2 < D / 16) get(n + 2);
    acc[n >> 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[n % 3], n & 1 ? x1 : x0, acc[n >> 1], 0, 0, 0);
    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
  }
}

template <int D, bool CAUSAL, int G>
__global__ void __launch_bounds__(512, 2) attn_bwd_dkdv_pair_kernel(FastBwdParams p) {
  constexpr int RW = 4, BK = 32 * RW, BQ = 32;
  constexpr int TILE = BQ * D * 2, KS = D / 16;
  // Q's tiles t - 1 (dK), t, and t + 1, t + 2 on their way; dO's t to t + 2; P of t - 1, t of each pair; lse and delta of t - 1 .. t + 1
  constexpr int NQ = 4, NG = 3;
  constexpr int GOFF = NQ * TILE, POFF = GOFF + NG * TILE, LOFF = POFF + 2 * RW * 4096;
  __shared__ __attribute__((aligned(1024))) char smem[LOFF + 4 * 64 * 4];
  static_assert(LOFF >= 2 * RW * TILE, "the epilogue's images take the tiles' place");

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), rw = wave % RW;
  const auto [kb, bh] = block_of<CAUSAL, D, BK>((p.Sk + BK - 1) / BK, p.B * p.Hkv);
  const int b = bh / p.Hkv, hk = bh % p.Hkv;
  const int grp = p.H / p.Hkv;
  const int off = p.Sk - p.Sq;
  const int kw = kb * BK + rw * 32;
  const int kv_end = batch_keys(p.kv_len, b, p.Sk);
  // what hangs on the lane is made anew where it is used, for the registers are full
  auto own_lane = [&] {
    int x = lane;
    asm volatile("" : "+v"(x));
    return x;
  };

  const int q_lo = CAUSAL ? max(0, kb * BK - off) & ~(BQ - 1) : 0;
  // no query sees a block past the length; past the last key's window no query sees the block
  const int q_end = p.window > 0 ? min(p.Sq, kb * BK + BK - 1 - off + p.window) : p.Sq;
  const int nqt = max(0, q_end - q_lo + BQ - 1) / BQ;
  const int total = kb * BK < kv_end ? nqt * grp : 0;
  // The walk goes from the last row back to the diagonal: the blocks of a head, which start together, read the same tiles together.
  const int q_top = q_lo + BQ * max(0, nqt - 1);
  float* const stat = reinterpret_cast<float*>(smem + LOFF);
  char* const pair = smem + POFF + rw * 4096;
  int be, b1, o_;
  row_bases<D>(lane & 31, lane >> 5, be, o_);
  tr_bases<D>(lane, b1, o_);

  f32x16 acc[D / 32];  // dV^T, or dK^T
  clear<D>(acc);
  bf16x8 fix[KS];  // K's rows, or V's
  auto load_fix = [&](const bf16_t* x, long long st) {
    const int key = kw + (lane & 31);
    const bf16_t* r = x + (long long)min(key, p.Sk - 1) * st + 8 * (lane >> 5);
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      fix[s] = *reinterpret_cast<const bf16x8*>(r + 16 * s);
      if (key >= kv_end) fix[s] = bf16x8{};
    }
  };

  if (wave < RW) {
    // The first waves request the tiles, two steps ahead: the second ones wait for loads of their own, which would wait for requests too.
    const float sl2 = p.scale * kLog2e;
    const int qn = rows_bytes(p.Sq, p.q_st, D), gn = rows_bytes(p.Sq, p.do_st, D);
    using Req = TileRequests<D, RW>;
    const Req lq(wave, lane, p.q_st), lg(wave, lane, p.do_st);
    const int stepq = BQ * (int)p.q_st * 2, stepg = BQ * (int)p.do_st * 2;
    const int soq0 = q_top * (int)p.q_st * 2, sog0 = q_top * (int)p.do_st * 2;
    // the tile being requested: first row, where it lies, query head (counted on: a step has no time to multiply)
    int qtr = q_top, soq = soq0, sog = sog0, headr = hk * grp;
    u32x4 rq, rg;
    auto words = [&] {
      rq = head_words(p.q + b * p.q_sb + headr * p.q_sh, qn), rg = head_words(p.dout + b * p.do_sb + headr * p.do_sh, gn);
    };
    auto next = [&] {
      qtr -= BQ, soq -= stepq, sog -= stepg;
      if (qtr >= q_lo) return;
      qtr = q_top, soq = soq0, sog = sog0, ++headr;
      words();
    };
    int sq = 0, sg = 0;  // their slots
    auto request = [&](int j) {
      if (j < Req::N) lq(rq, smem + sq * TILE, soq, j);
      else lg(rg, smem + GOFF + sg * TILE, sog, j - Req::N);
    };
    auto taken = [&] { sq = sq == NQ - 1 ? 0 : sq + 1, sg = sg == NG - 1 ? 0 : sg + 1; };
    if (total > 0) {  // (they fly with the key rows)
      words();
      auto tile = [&] {
#pragma unroll
        for (int j = 0; j < 2 * Req::N; ++j) request(j);
        taken();
      };
      tile();
      if (total > 1) next(), tile();
      load_fix(p.k + b * p.k_sb + hk * p.k_sh, p.k_st);
    }
    // The first tile is there. A tile that has none behind it is waited for with nothing else on its way, so that the walk's end waits for nothing.
    if (total > 1) wait_and_meet<2 * Req::N>();
    else wait_and_meet<0>();
    int qt = q_top, head = hk * grp, now = 0, at = 0;
    float slope = G == 2 ? p.alibi[head] * kLog2e : 0.f;
    auto step = [&](int i, auto more) {  // more: there is a tile to request
      if constexpr (more) next();
      asm volatile("" ::: "memory");
      const f32x16 s = pair_rows<D>(smem, now * TILE, be, fix, [&](int s) {
        if constexpr (more)
          if (s % 2 == 1) request(s / 2);
      });
      if constexpr (more) taken();
      const int ln = own_lane(), key = kw + (ln & 31), hh = ln >> 5;
      // rows q = qt + 8g + 4hh + j (g = r>>2, j = r&3) that see the key: lim <= 8g + j < ul
      const bool plain = kb * BK + BK <= kv_end && (!CAUSAL || kb * BK + BK - 1 <= qt + off) &&
                         (p.window <= 0 || kb * BK > qt + BQ - 1 + off - p.window);
      const float* ls = stat + (i & 3) * 64;
      const float b0 = slope * (float)(key - qt - off - 4 * hh);
      f32x16 pr;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 lq = *reinterpret_cast<const f32x4*>(ls + 8 * g + 4 * hh);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float bl = G == 2 ? fmaf(-slope, (float)(8 * g + j), b0) - lq[j] : -lq[j];
          pr[4 * g + j] = __builtin_amdgcn_exp2f(fmaf(s[4 * g + j], sl2, bl));
        }
      }
      if (!plain) {
        int lim = CAUSAL ? key - qt - off - 4 * hh : -(1 << 30);
        if (key >= kv_end) lim = 1 << 30;
        const int ul = p.window > 0 ? key + p.window - off - qt - 4 * hh : 1 << 30;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int c = 8 * (r >> 2) + (r & 3);
          if (c < lim || c >= ul) pr[r] = 0.f;
        }
      }
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<f32x4*>(pair + ln * 16 + (i & 1) * RW * 4096 + g * 1024) = f32x4{pr[4 * g], pr[4 * g + 1], pr[4 * g + 2], pr[4 * g + 3]};
      bf16x8 p0, p1;
#pragma unroll
      for (int r = 0; r < 8; ++r) p0[r] = (__bf16)pr[r], p1[r] = (__bf16)pr[r + 8];
      asm volatile("" ::: "memory");
      pair_columns<D>(acc, smem, GOFF + at * TILE, b1, p0, p1);
      now = now == NQ - 1 ? 0 : now + 1, at = at == NG - 1 ? 0 : at + 1;
      qt -= BQ;
      if (qt < q_lo) {
        qt = q_top, ++head;
        if (G == 2 && i + 1 < total) slope = p.alibi[head] * kLog2e;
      }
      wait_and_meet<more ? 2 * Req::N : 0>();  // the next tile is there
    };
    int i = 0;
    for (; i + 2 < total; ++i) step(i, std::true_type{});
    for (; i < total; ++i) step(i, std::false_type{});
    __syncthreads();  // the tiles become the epilogue images
    store_tile_lds<D, D, true>(p.dv + b * p.dv_sb + hk * p.dv_sh + (long long)kw * p.dv_st, p.dv_st, acc, lane, 1.f, smem + wave * TILE,
                               p.Sk - kw);
  } else {
    // lse and delta are the first two of the second waves' to bring; as they come: the scaling waits until they are stored
    const bool stats = rw < 2;
    int qt = q_top;
    const float* statp = (rw == 0 ? p.lse : p.delta) + ((long long)b * p.H + hk * grp) * p.Sq;
    auto next_stats = [&] {
      qt -= BQ;
      if (qt < q_lo) qt = q_top, statp += p.Sq;
    };
    auto load_stats = [&] { return stats ? statp[min(qt + (own_lane() & 31), p.Sq - 1)] : 0.f; };
    auto put_stats = [&](float x, int i) {
      if (stats) {
        const int sl = own_lane() & 31;
        float v = rw == 0 ? x * kLog2e : x;
        if (qt + sl >= p.Sq) v = rw == 0 ? INFINITY : 0.f;  // P = 0
        stat[(i & 3) * 64 + rw * 32 + sl] = v;              // (both halves of the wave alike)
      }
    };
    if (total > 0) {
      const float x = load_stats();
      load_fix(p.v + b * p.v_sb + hk * p.v_sh, p.v_st);
      put_stats(x, 0);
    }
    // what stands for the tile before the first: P = 0
#pragma unroll
    for (int g = 0; g < 4; ++g) *reinterpret_cast<f32x4*>(pair + lane * 16 + RW * 4096 + g * 1024) = f32x4{0.f, 0.f, 0.f, 0.f};
    if (rw == 1) stat[3 * 64 + lane] = 0.f;
    __syncthreads();
    int slot = 0, before = 0, at = 0;  // slots of tile i and the previous one (at first its own: P is 0), and of dO's
    f32x16 dp;
#pragma unroll
    for (int r = 0; r < 16; ++r) dp[r] = 0.f;
    for (int i = 0; i < (total > 0 ? total + 1 : 0); ++i) {
      const int ln = own_lane(), hh = ln >> 5;
      const float* ds = stat + ((i - 1) & 3) * 64 + 32;
      bf16x8 s0, s1;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 dl = *reinterpret_cast<const f32x4*>(ds + 8 * g + 4 * hh);
        const f32x4 pr = *reinterpret_cast<const f32x4*>(pair + ln * 16 + ((i - 1) & 1) * RW * 4096 + g * 1024);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float x = pr[j] * (dp[4 * g + j] - dl[j]);
          if (g < 2) s0[4 * g + j] = (__bf16)x;
          else s1[4 * g + j - 8] = (__bf16)x;
        }
      }
      asm volatile("" ::: "memory");
      if (i + 1 < total) next_stats();
      const float x = load_stats();
      pair_columns<D>(acc, smem, before * TILE, b1, s0, s1);
      before = slot;
      if (i < total) {
        dp = pair_rows<D>(smem, GOFF + at * TILE, be, fix);
        asm volatile("" ::: "memory");
        slot = slot == NQ - 1 ? 0 : slot + 1, at = at == NG - 1 ? 0 : at + 1;
        put_stats(x, i + 1);
        __syncthreads();
      }
    }
    __syncthreads();
    store_tile_lds<D, D, true>(p.dk + b * p.dk_sb + hk * p.dk_sh + (long long)kw * p.dk_st, p.dk_st, acc, lane, p.scale, smem + wave * TILE,
                               p.Sk - kw);
  }
}

template <int D, bool CAUSAL, int G>
__global__ void __launch_bounds__(512, 2) attn_bwd_dq_pair_kernel(FastBwdParams p) {
  constexpr int RW = 4, BM = 32 * RW, BN = 32;
  constexpr int TILE = BN * D * 2, KS = D / 16;
  // K's tiles t - 1 (dQ), t, and t + 1, t + 2 on their way; V's t to t + 2; P of t - 1, t of each pair
  constexpr int NK = 4, NV = 3;
  constexpr int VOFF = NK * TILE, POFF = VOFF + NV * TILE;
  __shared__ __attribute__((aligned(1024))) char smem[POFF + 2 * RW * 4096];

  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), rw = wave % RW;
  const int nqb = (p.Sq + BM - 1) / BM;
  const auto [qi, bh] = block_of<CAUSAL, D, BM>(nqb, p.B * p.H);
  const int qb = CAUSAL ? nqb - 1 - qi : qi;
  const int b = bh / p.H, h = bh % p.H, hk = h / (p.H / p.Hkv);
  const int off = p.Sk - p.Sq;
  const int q0 = qb * BM + rw * 32, qrow = q0 + l32, qr = min(qrow, p.Sq - 1);
  const int kv_end = batch_keys(p.kv_len, b, p.Sk);
  const TileSpan sp = tile_span<BM, CAUSAL>(qb * BM, off, kv_end, p.window);
  const int n = sp.hi - sp.lo;
  const long long li = ((long long)b * p.H + h) * p.Sq + qr;
  char* const pair = smem + POFF + rw * 4096 + lane * 16;
  int be, b1, o_;
  row_bases<D>(l32, hh, be, o_);
  tr_bases<D>(lane, b1, o_);

  auto on = [](int& slot, int slots) { slot = slot == slots - 1 ? 0 : slot + 1; };
  bf16x8 fix[KS];  // the rows of Q, or of dO
  if (wave < RW) {
    using Req = TileRequests<D, RW>;
    const Req lk(wave, lane, p.k_st), lv(wave, lane, p.v_st);
    const u32x4 kw = head_words(p.k + b * p.k_sb + hk * p.k_sh, rows_bytes(kv_end, p.k_st, D));
    const u32x4 vw = head_words(p.v + b * p.v_sb + hk * p.v_sh, rows_bytes(kv_end, p.v_st, D));
    const int stepk = BN * (int)p.k_st * 2, stepv = BN * (int)p.v_st * 2;
    int sok = sp.lo * stepk, sov = sp.lo * stepv, sk = 0, sv = 0;  // the tile being requested, two steps ahead, and its slots
    auto request = [&](int j) {
      if (j < Req::N) lk(kw, smem + sk * TILE, sok, j);
      else lv(vw, smem + VOFF + sv * TILE, sov, j - Req::N);
    };
    auto tile = [&] {
#pragma unroll
      for (int j = 0; j < 2 * Req::N; ++j) request(j);
      on(sk, NK), on(sv, NV), sok += stepk, sov += stepv;
    };
    tile();
    if (n > 1) tile();
    const bf16_t* qp = p.q + b * p.q_sb + h * p.q_sh + (long long)qr * p.q_st + 8 * hh;
#pragma unroll
    for (int s = 0; s < KS; ++s) fix[s] = *reinterpret_cast<const bf16x8*>(qp + 16 * s);
    const float sl2 = p.scale * kLog2e, nlse = -p.lse[li] * kLog2e, slope = G == 2 ? p.alibi[h] * kLog2e : 0.f;
    if (n > 1) wait_and_meet<2 * Req::N>();  // the first tile is there (as in dK/dV)
    else wait_and_meet<0>();
    int now = 0;
    auto step = [&](int i, auto more) {
      const int t = sp.lo + i, k0 = t * BN;
      asm volatile("" ::: "memory");
      const f32x16 s = pair_rows<D>(smem, now * TILE, be, fix, [&](int s) {
        if constexpr (more)
          if (s % 2 == 1) request(s / 2);
      });
      on(now, NK);
      if constexpr (more) on(sk, NK), on(sv, NV), sok += stepk, sov += stepv;
      const float b0 = G == 2 ? fmaf(slope, (float)(k0 + 4 * hh - qrow - off), nlse) : nlse;
      f32x16 pr;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int c = (r & 3) + 8 * (r >> 2);
        pr[r] = __builtin_amdgcn_exp2f(fmaf(s[r], sl2, G == 2 ? fmaf(slope, (float)c, b0) : b0));
      }
      if (t < sp.f_lo || t > sp.f_hi) {
        // visible key offsets: lo < offset <= lim
        const int lim = (CAUSAL ? min(qrow + off, kv_end - 1) : kv_end - 1) - k0 - 4 * hh;
        const int lo = p.window > 0 ? qrow + off - p.window - k0 - 4 * hh : -(1 << 30);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int c = (r & 3) + 8 * (r >> 2);
          if (c > lim || c <= lo) pr[r] = 0.f;
        }
      }
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<f32x4*>(pair + (i & 1) * RW * 4096 + g * 1024) = f32x4{pr[4 * g], pr[4 * g + 1], pr[4 * g + 2], pr[4 * g + 3]};
      wait_and_meet<more ? 2 * Req::N : 0>();  // the next tile is there
    };
    int i = 0;
    for (; i + 2 < n; ++i) step(i, std::true_type{});
    for (; i < n; ++i) step(i, std::false_type{});
    __syncthreads();  // the second waves' last step reads the tiles
    return;
  }
  f32x16 dq[D / 32];
  clear<D>(dq);
  const bf16_t* gp = p.dout + b * p.do_sb + h * p.do_sh + (long long)qr * p.do_st + 8 * hh;
  const bf16_t* op = p.o + b * p.o_sb + h * p.o_sh + (long long)qr * p.o_st + 8 * hh;
  float dl = 0.f;
#pragma unroll
  for (int s = 0; s < KS; ++s) fix[s] = *reinterpret_cast<const bf16x8*>(gp + 16 * s);
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const bf16x8 of = *reinterpret_cast<const bf16x8*>(op + 16 * s);
#pragma unroll
    for (int j = 0; j < 8; ++j) dl = fmaf((float)of[j], (float)fix[s][j], dl);
  }
  dl += __shfl_xor(dl, 32, 64);
  if (hh == 0 && qrow < p.Sq) p.delta[li] = dl;
  // what stands for the tile before the first: P = 0
#pragma unroll
  for (int g = 0; g < 4; ++g) *reinterpret_cast<f32x4*>(pair + RW * 4096 + g * 1024) = f32x4{0.f, 0.f, 0.f, 0.f};
  __syncthreads();
  int slot = 0, before = 0, at = 0;
  f32x16 dp;
#pragma unroll
  for (int r = 0; r < 16; ++r) dp[r] = 0.f;
  for (int i = 0; i <= n; ++i) {
    bf16x8 s0, s1;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 pr = *reinterpret_cast<const f32x4*>(pair + ((i - 1) & 1) * RW * 4096 + g * 1024);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float x = pr[j] * (dp[4 * g + j] - dl);
        if (g < 2) s0[4 * g + j] = (__bf16)x;
        else s1[4 * g + j - 8] = (__bf16)x;
      }
    }
    asm volatile("" ::: "memory");
    pair_columns<D>(dq, smem, before * TILE, b1, s0, s1);
    before = slot;
    if (i < n) {
      dp = pair_rows<D>(smem, VOFF + at * TILE, be, fix);
      asm volatile("" ::: "memory");
      on(slot, NK), on(at, NV);
      __syncthreads();
    }
  }
  __syncthreads();
  store_tile_lds<D, D, true>(p.dq + b * p.dq_sb + h * p.dq_sh + (long long)q0 * p.dq_st, p.dq_st, dq, lane, p.scale, smem + rw * TILE,
                             p.Sq - q0);
}

}  // namespace

// The backward of 256-wide heads whose rows are 16-byte aligned; 1: another call.
int attn_bwd_pair(const FastBwdParams& p, int d, bool causal, hipStream_t stream) {
  if (d != 256 || (p.alibi && !causal)) return 1;
  const dim3 gq((unsigned)((p.Sq + 127) / 128 * p.B * p.H)), gk((unsigned)((p.Sk + 127) / 128 * p.B * p.Hkv)), block(512);
  auto go = [&](auto C_, auto G_) {
    constexpr bool C = decltype(C_)::value;
    constexpr int G = decltype(G_)::value;
    hipLaunchKernelGGL((attn_bwd_dq_pair_kernel<256, C, G>), gq, block, 0, stream, p);
    hipLaunchKernelGGL((attn_bwd_dkdv_pair_kernel<256, C, G>), gk, block, 0, stream, p);
  };
  if (p.alibi) go(std::true_type{}, std::integral_constant<int, 2>{});
  else if (causal) go(std::true_type{}, std::integral_constant<int, 1>{});
  else go(std::false_type{}, std::integral_constant<int, 1>{});
  return hipGetLastError() == hipSuccess ? 0 : 3;
}
