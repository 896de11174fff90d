// What the matrix-core attention kernels of attention_tiled.hip, attention_split.hip and attention_pair.hip share: their parameters, the
// order of the blocks, the span of key tiles that a workgroup walks, fragment reads of a tile image, and the store of a wave's accumulator.
#pragma once
#include "attn_tile.h"

struct FastFwdParams {
  const bf16_t* q; const bf16_t* k; const bf16_t* v;
  bf16_t* o; float* lse;
  int* flags;  // [grid * 4]: 1 = this wave's rows overflowed -> fixup kernel
  long long q_sb, q_st, q_sh, k_sb, k_st, k_sh, v_sb, v_st, v_sh;
  long long o_sb, o_st, o_sh;
  int B, Sq, Sk, H, Hkv;
  float scale;
  const float* alibi;  // [H] slopes (G = 2)
  const int* kv_len;   // [B] or null (G > 0)
  int window;          // > 0: key visible only if key > q + off - window (G > 0)
  const int* cu;       // [B + 1] or null (G > 0): packed sequences -- batch b is rows cu[b] .. cu[b + 1], the batch
                       // strides are 0, Sq is the longest's length and lse null
};

__device__ __forceinline__ void own_sequence(FastFwdParams& p, int b) {
  const int c0 = p.cu[b];
  p.Sq = p.Sk = p.cu[b + 1] - c0;
  p.q += c0 * p.q_st;
  p.k += c0 * p.k_st;
  p.v += c0 * p.v_st;
  p.o += c0 * p.o_st;
}

// Which block (counted from the longest under a causal mask) of which head a workgroup takes. Causal: the longest blocks of all
// heads first, so that no long one starts when the others are done (heads a multiple of 8 also stay on their XCD): 2 x 2048 x 16
// heads of 256, whose 512 backward workgroups are two a CU, one after the other, 398 -> 298 us against head after head, 8 x 512
// of them with lengths 168 -> 129. Without a mask all are alike, and a head's blocks lie on one XCD, beside its keys and values.
// PER_CU: workgroups that run on a CU at one time. They start together, a round of 256 after the other, so that the CU with the longest
// block of the first round had the longest of the next as well: the later rounds are turned so that a CU's blocks add up to about the
// same (two: the second backwards; three: the second from its middle on, the third in twos backwards). 64-wide heads, 3 a CU, us,
// forward, dQ, dK/dV: 8 x 1000 x 12 heads 29.0, 36.0, 49.5 -> 26.7, 33.8, 46.4; 3 x 2048 x 16 46.7, 60.6, 91.3 -> 43.2, 56.9, 86.7. Two a
// CU (96 and 128 wide) gain or lose 3 %: not there.
//
// Many blocks: then the keys and values of all heads are walked at one time, and no cache holds them. An XCD takes its heads in turn, a
// head's blocks beside each other, and longest first among the last 1024 blocks alone (heads_in_turn). us, forward and backward, head after
// head, all heads at once, so: 559 tokens, 640 heads of 256 229, 275, 207 and 827, 814, 728; 300, 1280 of 256 236, 257, 185 and 740,
// 736, 644; 850, 1280 of 96 386, 464, 382 and 1053, 1178, 1025; 300, 640 of 128 57, 63, 57 and 174, 170, 161; 559, 640 of 64 71, 77, 70 and
// 214, 200, 188; 16 x 2048 x 16 of 256 634, 642, 607 and 2502, 2471, 2189. Where a head has 2, 4 or 8 blocks a CU meets one length
// again and again: 256 tokens, 1024 heads of 256 418, 463 in turn, 450 tokens, 1280 of 64 110, 117. Heads of 96 and 160 share 128-byte
// lines with their neighbours, which then lie on one XCD: short ones are taken so from the first block on (96: 128 tokens, 2048 heads 51,
// 47 and 147, 138; 300, 640 heads 59, 54; 2048, 128 heads 147, 156).
// (blocks of 128 rows: of a head, of all)
template <int D>
__device__ __forceinline__ bool heads_in_turn(int blocks, int total) {
  if (total > 8192 && blocks > 1) return true;
  if (D % 64) return blocks <= 10 || total > 3072;
  return blocks > 2 && (blocks % 4 || blocks > 8) && total > (blocks < 8 ? 1536 : 3072);
}
struct BlockOf { int block, head; };
template <bool CAUSAL, int D, int ROWS, int PER_CU = 1>
__device__ __forceinline__ BlockOf block_of(int blocks, int heads) {
  if (CAUSAL) {
    int n = (int)blockIdx.x;
    if (heads_in_turn<D>((blocks * ROWS + 127) / 128, (int)(gridDim.x * (long long)ROWS / 128))) {
      const int rest = heads % 8, own = heads / 8;  // (the heads that no XCD has for itself come first)
      if (n < rest * blocks) return {n / rest, 8 * own + n % rest};
      n -= rest * blocks;
      const int last = min(own, (128 + blocks - 1) / blocks), first = own - last, h0 = n % 8 * own;
      n /= 8;
      if (n < first * blocks) return {n % blocks, h0 + n / blocks};
      n -= first * blocks;
      return {n / last, h0 + first + n % last};
    }
    if constexpr (PER_CU == 3) {
      const int full = min(PER_CU, (int)gridDim.x / 256), round = n / 256, c = n / 8 % 32;  // (c: the CU of its XCD n % 8)
      if (round > 0 && round < full) {
        const int d = full == 2 ? 31 - c : round == 1 ? (c + 16) % 32 : c < 16 ? 31 - 2 * c : 62 - 2 * c;
        n = round * 256 + d * 8 + n % 8;
      }
    }
    return {n / heads, n % heads};
  }
  const int id = xcd_remap(blockIdx.x, gridDim.x);
  return {id % blocks, id / blocks};
}

constexpr int kAllRows = 0x7fffffff;

// buffer resource over one (batch, head) slice; the base is workgroup-uniform (readfirstlane'd so
// the descriptor is provably scalar: no waterfall loop, T20). `bytes`: loads at or past it return zeros.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t head_rsrc(const bf16_t* b, int bytes = kAllRows) {
  const unsigned long long a = (unsigned long long)b;
  const unsigned long long au = ((unsigned long long)__builtin_amdgcn_readfirstlane((unsigned)(a >> 32)) << 32) |
                                (unsigned)__builtin_amdgcn_readfirstlane((unsigned)a);
  return __builtin_amdgcn_make_buffer_rsrc((void*)au, (short)0, __builtin_amdgcn_readfirstlane(bytes), 0x00020000);
}
// bytes of `rows` rows of D elements, `st` elements apart
__device__ __forceinline__ int rows_bytes(int rows, long long st, int D) {
  return rows > 0 ? (int)(((rows - 1) * st + D) * 2) : 0;
}

// The 32-key tiles of a workgroup's query rows [r0, r0 + BM) in the general forms: it walks tiles [lo, hi),
// of which [f_lo, f_hi] need no mask. A row's last visible key lies in a tile above f_hi. For a row's first one, f_lo counts
// EDGE more tiles: 1, f_lo > lo and it lies in a tile below f_lo or at the start of f_lo; 2, below f_lo. At least one tile,
// also where no key is visible (a length of 0): its mask gives zeros.
struct TileSpan { int lo, hi, f_lo, f_hi; };
template <int BM, bool CAUSAL, int EDGE = 0>
__device__ __forceinline__ TileSpan tile_span(int r0, int off, int kv_end, int window) {
  TileSpan s;
  s.hi = max(1, ((CAUSAL ? min(kv_end, r0 + BM + off) : kv_end) + 31) / 32);
  s.f_hi = (CAUSAL ? min(r0 + off, kv_end - 1) : kv_end - 1) / 32 - 1;
  s.lo = s.f_lo = 0;
  if (window > 0) {
    s.lo = min(s.hi - 1, max(0, r0 + off - window + 1) / 32);
    s.f_lo = max(0, r0 + BM + off - window + (EDGE < 2 ? 31 : 32)) / 32;
  }
  if (EDGE) s.f_lo = max(s.f_lo, s.lo + 1);
  return s;
}
__device__ __forceinline__ int batch_keys(const int* kv_len, int b, int Sk) {
  return kv_len ? max(0, min(Sk, kv_len[b])) : Sk;
}

// Epilogue through LDS (cdna_hip_programming.md T21): the wave's 32 x D accumulator tile (row =
// lane & 31) goes into a wave-private [32][D] bf16 LDS image -- 16-B chunks rotated by the row,
// so the per-lane 8-B writes and the row-contiguous 16-B reads are both conflict-free -- and every
// store instruction then writes two whole rows with 16-B stores, instead of 8-B stores that each
// touch 64 rows. `mul` is the lane's row scale. The LDS must be free (after the loop's barrier).
// EDGE: only the first `rows` rows exist.
template <int D, int DS = D, bool EDGE = false>
__device__ __forceinline__ void store_tile_lds(bf16_t* row0, long long st, const f32x16 (&acc)[D / 32], int lane,
                                               float mul, char* lds, int rows = 32) {
  constexpr int NCH = D / 8, RB = D * 2, NCS = DS / 8;  // NCS: stored chunks per row
  const int l32 = lane & 31, hh = lane >> 5;
#pragma unroll
  for (int db = 0; db < D / 32; ++db) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      uint2 w;
      w.x = pk_bf16(acc[db][4 * g] * mul, acc[db][4 * g + 1] * mul);
      w.y = pk_bf16(acc[db][4 * g + 2] * mul, acc[db][4 * g + 3] * mul);
      *reinterpret_cast<uint2*>(lds + l32 * RB + ((4 * db + g + l32) % NCH) * 16 + hh * 8) = w;
    }
  }
  asm volatile("" ::: "memory");  // the wave's LDS accesses execute in order: reads see its writes
  static_assert((32 * NCS) % 64 == 0, "whole-wave epilogue rounds");
#pragma unroll
  for (int j = 0; j < 32 * NCS / 64; ++j) {
    const int idx = j * 64 + lane, r = idx / NCS, c = idx % NCS;
    const uint4 v = *reinterpret_cast<const uint4*>(lds + r * RB + ((c + r) % NCH) * 16);
    if (!EDGE || r < rows) *reinterpret_cast<uint4*>(row0 + (long long)r * st + c * 8) = v;
  }
  asm volatile("" ::: "memory");
}

struct FastBwdParams {
  const bf16_t* q; const bf16_t* k; const bf16_t* v; const bf16_t* dout;
  bf16_t* dq; bf16_t* dk; bf16_t* dv;
  const float* lse; float* delta;
  long long q_sb, q_st, q_sh, k_sb, k_st, k_sh, v_sb, v_st, v_sh, do_sb, do_st, do_sh;
  long long dq_sb, dq_st, dq_sh, dk_sb, dk_st, dk_sh, dv_sb, dv_st, dv_sh;
  int B, Sq, Sk, H, Hkv;
  float scale;
  const float* alibi;  // as in FastFwdParams
  const int* kv_len;
  int window;
  const bf16_t* o;
  long long o_sb, o_st, o_sh;
};

// A operand (32 rows x 16 k) read by rows from an image: lane (row l32, half hh)
// takes chunk 2s+hh of its row. Returns the two per-lane bases (s even / odd).
template <int D>
__device__ __forceinline__ void row_bases(int l32, int hh, int& e, int& o) {
  const int xr = (l32 >> 2) & 3;
  e = (l32 >> 3) * 16 * D + 64 * (l32 & 7) + 16 * (hh ^ xr);
  o = (l32 >> 3) * 16 * D + 64 * (l32 & 7) + 16 * ((2 + hh) ^ xr);
}
// transposed A operand (32 columns x 16 permuted rows) from an image
template <int D>
__device__ __forceinline__ void tr_bases(int lane, int& b1, int& b2) {
  const int hh = lane >> 5, gi = lane & 15;
  const int c3 = 2 * ((lane >> 4) & 1) + ((gi & 3) >> 1);
  b1 = 64 * (4 * hh + (gi >> 2)) + 16 * (c3 ^ hh) + 8 * (gi & 1);
  b2 = 16 * D + 64 * (4 * hh + (gi >> 2)) + 16 * (c3 ^ hh ^ 2) + 8 * (gi & 1);
}
template <int D>
__device__ __forceinline__ bf16x8 tr_frag(const char* img, int b1, int b2, int s, int db) {
  return cat8(lds_tr4(img, b1 + 2 * s * 16 * D + 512 * db), lds_tr4(img, b2 + 2 * s * 16 * D + 512 * db));
}
template <int D>
__device__ __forceinline__ bf16x8 row_frag(const char* img, int be, int bo, int s) {
  return lds_b128(img, ((s & 1) ? bo : be) + 512 * (s >> 1));
}

// a wave's accumulators as fp32, lane-linear: what the groups hand over to the one that adds them up
template <int D>
__device__ __forceinline__ void put_partial(char* at, const f32x16 (&acc)[D / 32], int lane) {
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<f32x4*>(at + ((db * 4 + g) * 64 + lane) * 16) =
          f32x4{acc[db][4 * g], acc[db][4 * g + 1], acc[db][4 * g + 2], acc[db][4 * g + 3]};
}
template <int D>
__device__ __forceinline__ void add_partial(const char* at, f32x16 (&acc)[D / 32], int lane, float w) {
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(at + ((db * 4 + g) * 64 + lane) * 16);
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[db][4 * g + j] = fmaf(x[j], w, acc[db][4 * g + j]);
    }
}

// the words of head_rsrc's descriptor, for inline asm
__device__ __forceinline__ u32x4 head_words(const bf16_t* b, int bytes) {
  const unsigned long long a = (unsigned long long)b;
  return u32x4{(unsigned)__builtin_amdgcn_readfirstlane((unsigned)a), (unsigned)__builtin_amdgcn_readfirstlane((unsigned)(a >> 32) & 0xffff),
               (unsigned)__builtin_amdgcn_readfirstlane(bytes), 0x00020000};
}

// A 32-row x D tile that NW waves request from memory straight into an image in LDS, N requests of 1 KB a wave (64 chunks of 16 bytes in the
// image's order; what lies past the descriptor's bytes becomes zeros). Counted by vmcnt; in asm, for hipcc would let every read of LDS
// wait for all of them. Five wait states stand before the request: a vector instruction may have written its scalars (readfirstlane, a
// spilled scalar), and in asm nobody else keeps the distance.
template <int D, int NW>
struct TileRequests {
  static constexpr int N = D / 16 / NW;
  static_assert(N * NW * 16 == D, "whole requests");
  unsigned from_[N];
  unsigned at_;
  __device__ __forceinline__ TileRequests(int wave, int lane, long long st) {
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const int q = (wave * N + j) * 64 + lane, sub = q / 32, row = sub / (D / 32) * 8 + q % 32 / 4;
      const int ch = sub % (D / 32) * 4 + ((q & 3) ^ ((row >> 2) & 3));  // img_off's inverse
      from_[j] = (unsigned)((row * st + ch * 8) * 2);
    }
    at_ = wave * N * 1024;
  }
  __device__ __forceinline__ void operator()(const u32x4& words, char* image, int so, int j) const {  // request j
#if defined(__HIP_DEVICE_COMPILE__)
    const unsigned to = (unsigned)(size_t)(__attribute__((address_space(3))) char*)image + at_ + j * 1024;
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(__builtin_amdgcn_readfirstlane(to)),
                 "v"(from_[j]), "s"(words), "s"(so)
                 : "m0");
#elif defined(LDS_TRACE)  // (a host build that follows requests and accesses)
    lds_request(image + at_ + j * 1024 + threadIdx.x % 64 * 16);
#endif
  }
};

// All but the wave's last N requests have landed, its LDS reads are done, and so are all other waves'.
template <int N>
__device__ __forceinline__ void wait_and_meet() {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#elif defined(LDS_TRACE)
  lds_wait(N);
  __syncthreads();
#endif
}

template <int D>
__device__ __forceinline__ void clear(f32x16 (&acc)[D / 32]) {
#pragma unroll
  for (int i = 0; i < D / 32; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[i][r] = 0.f;
}
