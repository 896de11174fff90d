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
// first one, which has less to do.
//
// Backward, us, one wave and a pair: 2 x 2048 x 16 heads 300, 266; 1 x 2048 225, 184; 1 x 4096 522, 454; 4 x 1100 234, 198; 8 x 512
// with lengths 128, 108; 1 x 3000 with ALiBi 361, 285; 3 x 300 56, 46; 1 x 61 24.7, 21.8. A tile of dK/dV takes 3200 cycles now, of dQ
// 2740 (1536 in the matrix cores): the LDS reads of both waves, 2085 of the 3200, and what of a wave's own chain the other does not
// cover. No gain: deeper rings of fragments, wave priorities, a walk that touches tiles ahead, heads turned over the XCDs.
#include "attn_fast.h"

#include <type_traits>

namespace {

__device__ __forceinline__ u32x4 buf_b128(__amdgpu_buffer_rsrc_t r, int vo, int so) {
  const auto a = __builtin_amdgcn_raw_buffer_load_b128(r, vo, so, 0);
  return *reinterpret_cast<const u32x4*>(&a);
}

struct Nothing { __device__ void operator()(int) const {} };

// Rows of a tile image times a fixed operand, the reads two steps ahead of their product (pinned), `also(s)` between; the last NF
// fragments of the operand come from LDS (`far`, a lane's 16 bytes of each 1 KB).
template <int D, int NF = 0, class Also = Nothing>
__device__ __forceinline__ f32x16 pair_rows(const char* smem, int img, int be, const bf16x8 (&fix)[D / 16], const char* far = nullptr,
                                            Also also = {}) {
  constexpr int KS = D / 16;
  f32x16 x;
#pragma unroll
  for (int r = 0; r < 16; ++r) x[r] = 0.f;
  bf16x8 f[3], l[NF ? NF : 1];
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
      if (t >= KS - NF) {
        l[t - KS + NF] = *reinterpret_cast<const bf16x8*>(far + (t - KS + NF) * 1024);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
    }
    also(s);
    x = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[s % 3], s >= KS - NF ? l[max(0, s - KS + NF)] : fix[s], x, 0, 0, 0);
    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
  }
  return x;
}

// acc += a tile image's columns times (x0, x1), read like its rows
template <int D, class Also = Nothing>
__device__ __forceinline__ void pair_columns(f32x16 (&acc)[D / 32], const char* smem, int img, int b1, bf16x8 x0, bf16x8 x1, Also also = {}) {
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
    also(n);
    acc[n >> 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[n % 3], n & 1 ? x1 : x0, acc[n >> 1], 0, 0, 0);
    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
  }
}

// A tile by the first four waves: a wave's lanes take 8 chunks of 8 rows, 128 bytes of each and 1 KB in a row in the image; the next
// 8 rows lie 16 D bytes on, their low sub-chunk bits turned.
template <int D>
struct PairLoader {
  static_assert(D == 256, "four waves, 8 of 32 chunks each");
  int vo, step;  // first chunk's byte offset, 8 rows
  __device__ __forceinline__ PairLoader(int wave, int lane, long long st)
      : vo((int)(((lane >> 3) * st + (wave * 8 + (lane & 7)) * 8) * 2)), step(__builtin_amdgcn_readfirstlane((int)(8 * st * 2))) {}
  __device__ __forceinline__ void load(u32x4& x, __amdgpu_buffer_rsrc_t r, int so, int j) const { x = buf_b128(r, vo, so + j * step); }
  static __device__ __forceinline__ int image(int wave, int lane) { return img_off<D>(lane >> 3, wave * 8 + (lane & 7)); }
  static __device__ __forceinline__ void put(const u32x4 (&x)[4], char* smem, int at) {  // at: image + the thread's place in it
#pragma unroll
    for (int j = 0; j < 4; ++j) *reinterpret_cast<u32x4*>(smem + (at ^ (j % 2 * 32)) + j * 16 * D) = x[j];
  }
};

template <int D, bool CAUSAL, int G>
__global__ void __launch_bounds__(512, 2) attn_bwd_dkdv_pair_kernel(FastBwdParams p) {
  constexpr int RW = 4, BK = 32 * RW, BQ = 32;
  constexpr int TILE = BQ * D * 2, KS = D / 16;
  // Q's tiles t - 1 (dK), t, t + 1 (loads); dO's t, t + 1; P of t - 1, t of each pair; lse and delta of t - 1 .. t + 1; the last NL of
  // K's KS fragments, for which no register is left
  constexpr int NL = 4;
  constexpr int GOFF = 3 * TILE, POFF = GOFF + 2 * TILE, LOFF = POFF + 2 * RW * 4096, FOFF = LOFF + 4 * 64 * 4;
  __shared__ __attribute__((aligned(16))) char smem[FOFF + NL * RW * 1024];
  static_assert(FOFF + NL * RW * 1024 >= 2 * RW * TILE, "the epilogue's images take the tiles' place");

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
    // The first waves bring the tiles. A step stores Q of the next one, requested in the step before, among its first products,
    // requests dO of the next one among the rest and stores it behind its softmax, and requests Q of the one after under dV.
    const float sl2 = p.scale * kLog2e;
    const int qn = rows_bytes(p.Sq, p.q_st, D), gn = rows_bytes(p.Sq, p.do_st, D);
    const PairLoader<D> lq(wave, lane, p.q_st), lg(wave, lane, p.do_st);
    const int own = PairLoader<D>::image(wave, lane);
    const int soq0 = __builtin_amdgcn_readfirstlane(q_top * (int)p.q_st * 2), sog0 = __builtin_amdgcn_readfirstlane(q_top * (int)p.do_st * 2);
    // the tiles of Q and of dO being loaded: first row, where it lies, query head (counted on: a step has no time to multiply)
    int qtq = q_top, soq = soq0, headq = hk * grp, qtg = q_top, sog = sog0, headg = hk * grp;
    __amdgpu_buffer_rsrc_t rq = head_rsrc(p.q + b * p.q_sb + headq * p.q_sh, qn), rg = head_rsrc(p.dout + b * p.do_sb + headg * p.do_sh, gn);
    auto next_q = [&] {
      qtq -= BQ, soq -= 4 * lq.step;
      if (qtq >= q_lo) return;
      qtq = q_top, soq = soq0, ++headq;
      rq = head_rsrc(p.q + b * p.q_sb + headq * p.q_sh, qn);
    };
    auto next_g = [&] {
      qtg -= BQ, sog -= 4 * lg.step;
      if (qtg >= q_lo) return false;
      qtg = q_top, sog = sog0, ++headg;
      rg = head_rsrc(p.dout + b * p.do_sb + headg * p.do_sh, gn);
      return true;
    };
    u32x4 xq[4];
    if (total > 0) {  // (flies with the key rows)
      u32x4 xg[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) lq.load(xq[j], rq, soq, j), lg.load(xg[j], rg, sog, j);
      load_fix(p.k + b * p.k_sb + hk * p.k_sh, p.k_st);
#pragma unroll
      for (int s = KS - NL; s < KS; ++s) *reinterpret_cast<bf16x8*>(smem + FOFF + (rw * NL + s - KS + NL) * 1024 + lane * 16) = fix[s];
      PairLoader<D>::put(xq, smem, own);
      PairLoader<D>::put(xg, smem, GOFF + own);
      if (total > 1) next_q();
#pragma unroll
      for (int j = 0; j < 4; ++j) lq.load(xq[j], rq, soq, j);
    }
    __syncthreads();
    float next_slope = G == 2 ? p.alibi[headg] * kLog2e : 0.f;
    int slot = 0;  // of tile i in Q's three
    for (int i = 0; i < total; ++i) {
      const int qt = qtg;
      const float slope = next_slope;
      // (past the last tile a step loads it again, into the slots that nobody reads)
      if (i + 1 < total && next_g() && G == 2) next_slope = p.alibi[headg] * kLog2e;
      if (i + 2 < total) next_q();
      const int now = slot * TILE;
      slot = slot == 2 ? 0 : slot + 1;
      const int then = slot * TILE, at = GOFF + (i & 1) * TILE;
      u32x4 xg[4];
      asm volatile("" ::: "memory");
      const f32x16 s = pair_rows<D, NL>(smem, now, be, fix, smem + FOFF + rw * NL * 1024 + lane * 16, [&](int s) {
        if (s == 7) {
          PairLoader<D>::put(xq, smem, then + own);
          __builtin_amdgcn_sched_group_barrier(0x200, 4, 0);
        }
        if (s >= 8 && s % 2 == 0) {
          lg.load(xg[s / 2 - 4], rg, sog, s / 2 - 4);
          __builtin_amdgcn_sched_group_barrier(0x20, 1, 0);
        }
      });
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
      PairLoader<D>::put(xg, smem, GOFF + ((i + 1) & 1) * TILE + own);
      asm volatile("" ::: "memory");
      pair_columns<D>(acc, smem, at, b1, p0, p1, [&](int n) {
        if (n % 2 == 0 && n < 8) {
          lq.load(xq[n / 2], rq, soq, n / 2);
          __builtin_amdgcn_sched_group_barrier(0x20, 1, 0);
        }
      });
      __syncthreads();
    }
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
    int slot = 0, before = 0;  // slots of tile i and the previous one (at first its own: P is 0)
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
        dp = pair_rows<D>(smem, GOFF + (i & 1) * TILE, be, fix);
        asm volatile("" ::: "memory");
        slot = slot == 2 ? 0 : slot + 1;
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
  constexpr int VOFF = 3 * TILE, POFF = VOFF + 2 * TILE;  // K's tiles t - 1 (dQ), t, t + 1 (loads); V's t, t + 1; P of t - 1, t of each pair
  __shared__ __attribute__((aligned(16))) char smem[POFF + 2 * RW * 4096];

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

  bf16x8 fix[KS];  // the rows of Q, or of dO
  if (wave < RW) {
    const int kn = rows_bytes(kv_end, p.k_st, D), vn = rows_bytes(kv_end, p.v_st, D);
    const __amdgpu_buffer_rsrc_t rk = head_rsrc(p.k + b * p.k_sb + hk * p.k_sh, kn), rv = head_rsrc(p.v + b * p.v_sb + hk * p.v_sh, vn);
    const PairLoader<D> lk(wave, lane, p.k_st), lv(wave, lane, p.v_st);
    const int own = PairLoader<D>::image(wave, lane);
    // the tile being loaded, a step before it is stored and two before it is read
    int sok = __builtin_amdgcn_readfirstlane(sp.lo * 4 * lk.step), sov = __builtin_amdgcn_readfirstlane(sp.lo * 4 * lv.step);
    u32x4 xk[4], xv[4];
    auto load = [&] {
#pragma unroll
      for (int j = 0; j < 4; ++j) lk.load(xk[j], rk, sok, j), lv.load(xv[j], rv, sov, j);
    };
    load();
    const bf16_t* qp = p.q + b * p.q_sb + h * p.q_sh + (long long)qr * p.q_st + 8 * hh;
#pragma unroll
    for (int s = 0; s < KS; ++s) fix[s] = *reinterpret_cast<const bf16x8*>(qp + 16 * s);
    const float sl2 = p.scale * kLog2e, nlse = -p.lse[li] * kLog2e, slope = G == 2 ? p.alibi[h] * kLog2e : 0.f;
    PairLoader<D>::put(xk, smem, own);
    PairLoader<D>::put(xv, smem, VOFF + own);
    if (n > 1) sok += 4 * lk.step, sov += 4 * lv.step;
    load();
    __syncthreads();
    int slot = 0;  // of tile i in K's three
    for (int i = 0; i < n; ++i) {
      const int t = sp.lo + i, k0 = t * BN, now = slot * TILE;
      slot = slot == 2 ? 0 : slot + 1;
      const int then = slot * TILE;
      if (i + 2 < n) sok += 4 * lk.step, sov += 4 * lv.step;  // (past the last tile: it again, into slots that nobody reads)
      asm volatile("" ::: "memory");
      const f32x16 s = pair_rows<D>(smem, now, be, fix, nullptr, [&](int s) {
        if (s == 3 || s == 5) {
          if (s == 3) PairLoader<D>::put(xk, smem, then + own);
          else PairLoader<D>::put(xv, smem, VOFF + ((i + 1) & 1) * TILE + own);
          __builtin_amdgcn_sched_group_barrier(0x200, 4, 0);
        }
        if (s >= 8) {
          if (s % 2 == 0) lk.load(xk[s / 2 - 4], rk, sok, s / 2 - 4);
          else lv.load(xv[s / 2 - 4], rv, sov, s / 2 - 4);
          __builtin_amdgcn_sched_group_barrier(0x20, 1, 0);
        }
      });
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
      __syncthreads();
    }
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
  int slot = 0, before = 0;
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
      dp = pair_rows<D>(smem, VOFF + (i & 1) * TILE, be, fix);
      asm volatile("" ::: "memory");
      slot = slot == 2 ? 0 : slot + 1;
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
