// Expert products whose tiles the memory system brings straight into LDS: the weight stream of few rows and the wide blocks of prompts
// (moe.hip launches them), with their requests and waits, which a host build follows (LDS_TRACE).
#pragma once
#include "common.h"

namespace {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

struct ExpertArgs {
  const void* x;        // gate-up: [T][K] token rows; down: [n][K] sorted rows
  const void* w;        // [E][2N or N][K]
  void* y;              // [n][N] sorted rows
  const int* perm;
  const float* wts;     // [n] by assignment
  const int* tiles;
  const int* ntiles;
  int mt;               // row limit of a tile
  int top, N, K, up, scale;  // up: gate-and-up (x gathered by token, silu product); scale: the weight applies here
  // gemv: a shared expert beside them, `tokens` rows in order, without a weight (ws null: none)
  const void* xs;       // [tokens][Ks]
  const void* ws;       // [2Ns or Ns][Ks]
  void* ys;             // [tokens][Ns]
  int tokens, Ns, Ks;
};

// Whether the last tile of an expert with `c` rows stands after all experts' others (row limits of 128 and 192): it is at most half
// full, and what its weights cost to read again, away from the expert's other tiles, is less than the CUs that it fills: two full
// tiles before it, or none, or one of 192 rows and hardly any rows. Both products, us (width, experts, top, inner size), beside its
// expert's and last: 3000 tokens, 2048, 32, 4, 1024 237, 215; 300, 4096, 16, 3, 2048 218, 199.
__device__ __forceinline__ bool late_tile(int c, int mt) {
  const int r = c % mt, full = c / mt;
  return mt >= 128 && mt < 256 && r && 2 * r <= mt && (full != 1 || (mt > 128 && 8 * r <= mt));
}

// Whether a tile's weights come non-temporal (request_into_lds): no other tile reads them beside it or later. `tiles`: how many stand together. A
// late one is the last to read its expert's weights, but a full one of 192 rows by itself may have a late one after it, which finds them in the last
// cache (196 rows an expert, cold, us, both non-temporal, both ordinary, so: 24 experts of 3 x 2048 x 768 120, 104, 103.5; 32 of 3 x 2048 x 1024 210, 193,
// 179; 16 of 3 x 4096 x 2048 389, 375, 348; of 3 x 4096 x 4096 672, 677, 638).
// Tiles that stand together: in the gemm the second of two finds what the first has read: 24 experts of 3 x 2048 x 768, top 5, 500 tokens, us, ordinary
// 101.3, non-temporal all 102.2, so 97.3; 777 112.3, 114.4, 110.4; 16 of 3 x 4096 x 2048, top 3, 300 210.5, 192, 192.5; 777 267, 253, 250.6.
__device__ __forceinline__ bool read_once(int tiles, int rows, int mt) { return tiles == 1 && !(mt > 128 && rows == mt); }

// the words of a descriptor of everything from p on, for inline asm
__device__ __forceinline__ u32x4 uniform_words(const void* p) {
  const unsigned long long a = (unsigned long long)p;
  return u32x4{(unsigned)__builtin_amdgcn_readfirstlane((unsigned)a), (unsigned)__builtin_amdgcn_readfirstlane((unsigned)(a >> 32) & 0xffff), ~0u,
               0x00020000};
}


// A place's address as requests take it
__device__ __forceinline__ unsigned lds_address(const char* p) {
#if defined(LDS_TRACE)
  return lds_offset(p);
#else
  return (unsigned)(size_t)(__attribute__((address_space(3))) const char*)p;
#endif
}

// 16 bytes a lane, 1 KB in a row at `at`, from `from` + k bytes on. ONCE: non-temporal, for the weights of an expert that has one tile, which no other
// block reads. One layer, cold, us, without and with: 16 experts of 3 x 4096 x 4096, top 2, 32 tokens 300, 287 (stream, 5.6 TB/s), 100 308, 293; 777 372,
// 350 (wide blocks of up to 192 rows; those of 256, bound by the products, gain nothing: not there), 1200 406, 392; 3 x 4096 x 2048, top 3, 32 175, 166; 130 189, 177
// (blocks of 128 weight rows). (In asm: hipcc would let every read of LDS wait for all requests. Nothing is
// returned to a register. Five wait states after what may be a vector write of a scalar)
template <bool ONCE = false>
__device__ __forceinline__ void request_into_lds(const u32x4& rsrc, unsigned at, unsigned from, int k) {
#if defined(LDS_TRACE)
  lds_request_at(at + threadIdx.x % 64 * 16);
#else
  if constexpr (ONCE)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tbuffer_load_dwordx4 %1, %2, %3 offen nt lds" ::"s"(__builtin_amdgcn_readfirstlane(at)),
                 "v"(from), "s"(rsrc), "s"(k)
                 : "m0");
  else
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(__builtin_amdgcn_readfirstlane(at)),
                 "v"(from), "s"(rsrc), "s"(k)
                 : "m0");
#endif
}

// All of the wave's requests but its newest N have landed
template <int N>
__device__ __forceinline__ void wait_requests() {
#if defined(LDS_TRACE)
  lds_wait(N);
#else
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
#endif
}
// its reads of LDS as well
template <int N>
__device__ __forceinline__ void wait_requests_and_reads() {
#if defined(LDS_TRACE)
  lds_wait(N);
#else
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
#endif
}
__device__ __forceinline__ void wait_reads() {
#if !defined(LDS_TRACE)
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#endif
}

// ---------------------------------------------------------------------------------------------- stream
// bf16, tiles of up to 32 rows x 32 weight rows (up: 16 gate rows and the 16 up rows beside them), 4 waves, each with every fourth stage
// of 64 of K; the waves' sums meet in LDS. Bound by the weight stream. How fast memory gives it hangs on how far apart the rows lie that
// the chip reads at one time: blocks of 64 rows that walk K by themselves have the whole of a weight in flight, ordinary loads 4.7 to 4.9 TB/s (50432 x
// 4096, loads alone), of 32 rows, K over the waves, 6.0; the number of bytes in flight and the length of a request's rows make no
// difference. A wave's stages go straight to LDS, weights three stages ahead, activations, in the XCD's cache, two; no wave
// waits for another before the end, and two workgroups a CU cover each other's ramps. Beside the gemv kernel, whose vector products a row
// cost more than its weights from about 2 rows an expert on, and the gemm, which computes and stages mostly padding.
// Both products of a layer, us, ordinary loads, blocks of 64 weight rows that walk K by themselves (the form before) and this: 20 outputs, 16 experts of 3 x
// 4096 x 2048, top 3: 20 tokens 163, 142, 64 173, 143; 32 of 3 x 2048 x 1024, top 4: 64 85, 80; 16 of 3 x 4096 x 4096, top 2: 32 282,
// 274, 130 295, 278. Workgroups in plain order 149, 87, 281, 307; an XCD a contiguous eighth of the blocks 161, 84, 278, 301; runs of
// 512 151, 83, 293, 308; a fourth weight stage, one workgroup a CU, 172, 102, 285, 310.
// K % 64 == 0 and N % 16 == 0; an LDS-DMA instruction fills 8 rows of 128 bytes lane by lane, so the 16-byte pieces
// are swizzled (by row pair: 16 rows x one piece cover all 64 banks) on the source address.
constexpr int SROWS = 32, SK = 64, SWN = 32;

// rows: 8, 16 or 32 of activations (XI requests a stage)
template <bool UP, int XI, bool ONCE = false>
__device__ __forceinline__ void expert_stream_tile(const ExpertArgs& p, char* sl, int ex, int lo, int nr, int n0) {
  constexpr int XB = XI > 2 ? 2 : 1, NW = 3, NX = 2, OWN = NW * 4096 + NX * XI * 1024;  // runs of 16 rows; places; a wave's bytes
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, g = lane >> 4, K = p.K, N = p.N;
  const u32x4 rw = uniform_words(reinterpret_cast<const bf16_t*>(p.w) + (long long)ex * (UP ? 2 * N : N) * K);
  const u32x4 rx = uniform_words(reinterpret_cast<const bf16_t*>(p.x) + (UP ? 0ll : (long long)lo * K));
  unsigned wo[4], xo[XI];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 8 * i + (lane >> 3), n = UP ? (i < 2 ? 0 : N) + n0 + (r & 15) : min(n0 + r, N - 1);
    wo[i] = ((unsigned)n * K + 8 * ((lane & 7) ^ ((r >> 1) & 7))) * 2;
  }
#pragma unroll
  for (int i = 0; i < XI; ++i) {
    const int r = 8 * i + (lane >> 3), xr = min(r, nr - 1);
    xo[i] = ((unsigned)(UP ? p.perm[lo + xr] / p.top : xr) * K + 8 * ((lane & 7) ^ ((r >> 1) & 7))) * 2;
  }
  const int nk = K / SK, last = nk > wv ? (nk - 1 - wv) / 4 * 4 + wv : 0;  // the wave's last stage
  char* const own = sl + wv * OWN;
  const unsigned base = __builtin_amdgcn_readfirstlane(lds_address(own));
  auto stage_k = [&](int t) { return __builtin_amdgcn_readfirstlane(min(4 * t + wv, last) * SK * 2); };  // past the end: one that nobody reads
  auto weights = [&](int t, int place) {
#pragma unroll
    for (int i = 0; i < 4; ++i) request_into_lds<ONCE>(rw, base + place * 4096 + i * 1024, wo[i], stage_k(t));
  };
  auto rows = [&](int t, int place) {
#pragma unroll
    for (int i = 0; i < XI; ++i) request_into_lds(rx, base + NW * 4096 + (place * XI + i) * 1024, xo[i], stage_k(t));
  };
  f32x4 acc[2][XB];  // [gate, up | two runs of 16 outputs][16 rows]
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < XB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int sw = (r16 >> 1) & 7;
  rows(0, 0);
  weights(0, 0);
  rows(1, 1);
  weights(1, 1);
  weights(2, 2);
  int pw = 0, px = 0;
  for (int t = 0; 4 * t + wv < nk; ++t) {
    wait_requests<8 + XI>();  // stage t has landed; weights t + 1, t + 2 and rows t + 1 may be on their way
    bf16x8 a[2][2], x[2][XB];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int c = ((4 * s + g) ^ sw) * 16;
#pragma unroll
      for (int i = 0; i < 2; ++i) a[s][i] = *reinterpret_cast<const bf16x8*>(own + pw * 4096 + (16 * i + r16) * 128 + c);
#pragma unroll
      for (int j = 0; j < XB; ++j)  // (8 rows: twice)
        x[s][j] = *reinterpret_cast<const bf16x8*>(own + NW * 4096 + px * XI * 1024 + (16 * j + (XI == 1 ? r16 & 7 : r16)) * 128 +
                                                   ((4 * s + g) ^ (XI == 1 ? ((r16 & 7) >> 1) : sw)) * 16);
    }
    wait_reads();
    rows(t + 2, px);
    weights(t + 3, pw);
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < XB; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[s][i], x[s][j], acc[i][j], 0, 0, 0);
    pw = pw == NW - 1 ? 0 : pw + 1;
    px ^= 1;
  }
  wait_requests<0>();  // the repeated stages, before their places are used again
  __syncthreads();
  f32x4* const part = reinterpret_cast<f32x4*>(sl);  // [run][rows][wave][lane]
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < XB; ++j) part[((i * XB + j) * 4 + wv) * 64 + lane] = acc[i][j];
  __syncthreads();
  auto sum = [&](int i, int j) {  // in the order of the waves
    f32x4 s = part[(i * XB + j) * 256 + lane];
#pragma unroll
    for (int w = 1; w < 4; ++w) s += part[((i * XB + j) * 4 + w) * 64 + lane];
    return s;
  };
  if (wv >= (UP ? XB : 2 * XB)) return;
  const int j = UP ? wv : wv % XB, i = UP ? 0 : wv / XB, r = 16 * j + r16, n = n0 + 16 * i + 4 * g;
  if (r >= nr || n >= N) return;
  const float s = p.scale ? p.wts[p.perm[lo + r]] : 1.f;
  const f32x4 u = sum(i, j), v = UP ? sum(1, j) : u;
  float o[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if constexpr (UP) {
      const float gt = u[e] * s, up = v[e] * s;
      o[e] = gt * __builtin_amdgcn_rcpf(1.f + __expf(-gt)) * up;
    } else {
      o[e] = u[e] * s;
    }
  }
  bf16_t* y = reinterpret_cast<bf16_t*>(p.y) + (long long)(lo + r) * N;
  *reinterpret_cast<uint2*>(y + n) = make_uint2(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]));
}
constexpr int STREAM_LDS = 4 * (3 * 4096 + 2 * 4 * 1024);

// The same tiles x 128 weight rows (up: 64 gate rows and the 64 up rows beside them) that walk K by themselves, 32 of them a wave; all waves read a
// stage's activations, requested once: 20 KB a stage, three stages ahead, two workgroups a CU. It has a quarter of the blocks, starts and
// sums over waves, and half as many requests a weight row where tiles have more than 16 rows, but its weights come slower (ordinary loads 4.7 to 4.9 TB/s). So it is the
// better one where the walk is short for its rows (stream_block).
constexpr int BWN = 128, BSTAGE = (BWN + SROWS) * SK * 2;
static_assert(4 * BSTAGE == STREAM_LDS, "four stages");
template <bool UP, bool ONCE = false>
__device__ __forceinline__ void expert_block_tile(const ExpertArgs& p, char* sl, int ex, int lo, int nr, int n0) {
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, g = lane >> 4, K = p.K, N = p.N, nk = K / SK;
  const u32x4 rw = uniform_words(reinterpret_cast<const bf16_t*>(p.w) + (long long)ex * (UP ? 2 * N : N) * K);
  const u32x4 rx = uniform_words(reinterpret_cast<const bf16_t*>(p.x) + (UP ? 0ll : (long long)lo * K));
  // a wave requests its own 32 weight rows and 8 of the activations'
  unsigned wo[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 8 * i + (lane >> 3), n = UP ? (i < 2 ? 0 : N) + min(n0 + wv * 16 + (r & 15), N - 1) : min(n0 + wv * 32 + r, N - 1);
    wo[i] = ((unsigned)n * K + 8 * ((lane & 7) ^ ((r >> 1) & 7))) * 2;
  }
  const int xr = wv * 8 + (lane >> 3), row = min(xr, nr - 1);
  const unsigned xo = ((unsigned)(UP ? p.perm[lo + row] / p.top : row) * K + 8 * ((lane & 7) ^ ((xr >> 1) & 7))) * 2;
  const unsigned base = __builtin_amdgcn_readfirstlane(lds_address(sl));
  auto request = [&](int t) {
    const int k = __builtin_amdgcn_readfirstlane(min(t, nk - 1) * SK * 2);  // past the end: the last one, which nobody reads
    const unsigned at = base + t % 4 * BSTAGE;
#pragma unroll
    for (int i = 0; i < 4; ++i) request_into_lds<ONCE>(rw, at + (wv * 4 + i) * 1024, wo[i], k);
    request_into_lds(rx, at + (16 + wv) * 1024, xo, k);
  };
  f32x4 acc[2][2];  // [gate, up | two runs of 16 outputs][16 rows]
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int sw = (r16 >> 1) & 7;
#pragma unroll
  for (int t = 0; t < 3; ++t) request(t);
  for (int t = 0; t < nk; ++t) {
    wait_requests_and_reads<10>();  // the wave's pieces of stage t have landed and it has read stage t - 1; so have all others'
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    request(t + 3);  // where stage t - 1 was
    const char* const st = sl + t % 4 * BSTAGE;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int c = ((4 * s + g) ^ sw) * 16;
      bf16x8 a[2], x[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) a[i] = *reinterpret_cast<const bf16x8*>(st + (wv * 32 + 16 * i + r16) * 128 + c);
#pragma unroll
      for (int j = 0; j < 2; ++j) x[j] = *reinterpret_cast<const bf16x8*>(st + (BWN + 16 * j + r16) * 128 + c);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], x[j], acc[i][j], 0, 0, 0);
    }
  }
  wait_requests<0>();  // the repeated stages, before the LDS is given back
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int r = 16 * j + r16;
    if (r >= nr) continue;
    const float s = p.scale ? p.wts[p.perm[lo + r]] : 1.f;
    bf16_t* y = reinterpret_cast<bf16_t*>(p.y) + (long long)(lo + r) * N;
#pragma unroll
    for (int i = 0; i < (UP ? 1 : 2); ++i) {
      const int n = n0 + wv * (UP ? 16 : 32) + 16 * i + 4 * g;
      if (n >= N) continue;
      float o[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (UP) {
          const float gt = acc[0][j][e] * s, up = acc[1][j][e] * s;
          o[e] = gt * __builtin_amdgcn_rcpf(1.f + __expf(-gt)) * up;
        } else {
          o[e] = acc[i][j][e] * s;
        }
      }
      *reinterpret_cast<uint2*>(y + n) = make_uint2(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]));
    }
  }
}

// ------------------------------------------------------------------------------------------------ turns
constexpr int GBK = 64, GN = 256, GM = 256, GEMM_LDS = 2 * (GN + GM) * GBK * 2, WIDE_LDS = GEMM_LDS / 4 * 5;

// Wide blocks where K % 64 == 0: 8 waves in two groups of four, one of each on a SIMD. While one group multiplies, the other reads its
// next fragments from LDS and requests stages, and a barrier later they change places, so that a SIMD's matrix core always has a wave that
// does nothing else. (4 waves of 128 x 128, a wave alone on its SIMD, whose products waited for its loads, barriers and issue: 59 % of
// a block's time multiplied. Here 92 % of the loop, 80 % of a block; 142 thousand cycles for 64 stages of 256 rows, 131 the products alone.)
// A group holds half of the block's weight rows (128: two halves of 64; up: gate rows and their up rows), a wave of it a quarter of the
// rows, in B runs of 16: 64 B rows a tile. A turn is one half of the weight rows over a stage of 64 of K: 8 B products of 16x16x32 after 8
// fragments of weights and, first half, 2 B of activations, which the second half multiplies again.
// Stages go straight into LDS in whole 128-byte lines (a request: 8 rows, 16-byte pieces swizzled by row pair on the source address, so 16
// rows x one piece cover all 64 banks). Weights have three places and are requested two stages ahead; activations, hit in the XCD's cache
// more often, two places, requested as soon as both groups have read the first half. A turn between products must be shorter than one of
// products: LDS reads and requests alternate, since each kind alone holds a wave up while the other's path is idle (all reads first 147
// thousand cycles; requests between the products, which then wait for the address path, 208).
// A whole sublayer, us, this and four waves before: 4096 tokens, 16 experts of 3 x 4096 x 4096, top 2 882 -> 774, with another routing 969 ->
// 810; 2000 tokens 589 -> 482, 1200 412 -> 386; 4000 tokens, 16 of 3 x 4096 x 2048, top 3 574 -> 481.
// What bounds it: rounds of blocks that end half empty (15 % at 4096 tokens), a block's start and results (22 thousand cycles). Blocks
// that stay and request the next tile before their results gained nothing over the scheduler's choice of the next block.
template <bool UP, int B, bool ONCE = false>
__device__ __forceinline__ void expert_turns_tile(const ExpertArgs& p, char* sl, int ex, int lo, int nr, int n0) {
  constexpr int HALF = 128 * GBK * 2, BST = 64 * B * GBK * 2, BAT = 6 * HALF;  // bytes: 128 weight rows, the activations of a stage, their place
  static_assert(BAT + 2 * BST <= WIDE_LDS, "three stages of weights and two of activations");
  const int tid = threadIdx.x, lane = tid & 63, r16 = lane & 15, g = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), wa = wv >> 2, wb = wv & 3;  // wa: the group
  const int K = p.K, N = p.N, nk = K / GBK;
  const u32x4 rw = uniform_words(reinterpret_cast<const bf16_t*>(p.w) + (long long)ex * (UP ? 2 * N : N) * K);
  const u32x4 rx = uniform_words(reinterpret_cast<const bf16_t*>(p.x) + (UP ? 0ll : (long long)lo * K));
  unsigned from_w[4], from_x[B];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = (wb * 4 + i) * 8 + (lane >> 3);  // of the half's 128: 64 of either group
    const int n = UP ? wa * N + min(n0 + r, N - 1) : min(n0 + (r >> 6) * 128 + wa * 64 + (r & 63), N - 1);
    from_w[i] = ((unsigned)n * K + 8 * ((lane & 7) ^ ((r >> 1) & 7))) * 2;
  }
#pragma unroll
  for (int i = 0; i < B; ++i) {
    const int r = (wv * B + i) * 8 + (lane >> 3), xr = min(r, nr - 1);
    from_x[i] = ((unsigned)(UP ? p.perm[lo + xr] / p.top : xr) * K + 8 * ((lane & 7) ^ ((r >> 1) & 7))) * 2;
  }
  const unsigned base = __builtin_amdgcn_readfirstlane(lds_address(sl));
  auto request = [&](auto once, const u32x4& rsrc, unsigned at, unsigned from, int t) {
    request_into_lds<decltype(once)::value>(rsrc, at, from, __builtin_amdgcn_readfirstlane(min(t, nk - 1) * GBK * 2));  // past the end: the last one, which nobody reads
  };
  auto weight = [&](int t, int place, int i) { request(std::integral_constant<bool, ONCE>{}, rw, base + (2 * place + wa) * HALF + (wb * 4 + i) * 1024, from_w[i], t); };
  auto row = [&](int t, int place, int i) { request(std::false_type{}, rx, base + BAT + place * BST + (wv * B + i) * 1024, from_x[i], t); };
  f32x4 acc[2][4][B];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < B; ++j) acc[h][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  bf16x8 a[2][4], x[2][B];
  const int sw = (r16 >> 1) & 7, ar = (wa * 64 + r16) * 128, xr = BAT + (wb * 16 * B + r16) * 128;
  auto read_w = [&](int place, int h, int s, int i) {
    a[s][i] = *reinterpret_cast<const bf16x8*>(sl + (2 * place + h) * HALF + ar + ((4 * s + g) ^ sw) * 16 + i * 2048);
  };
  auto read_x = [&](int place, int s, int j) { x[s][j] = *reinterpret_cast<const bf16x8*>(sl + place * BST + xr + ((4 * s + g) ^ sw) * 16 + j * 2048); };
  auto change = [&] {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  auto products = [&](int h) {
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < B; ++j) acc[h][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[s][i], x[s][j], acc[h][i][j], 0, 0, 0);
    __builtin_amdgcn_s_setprio(0);
  };
#pragma unroll
  for (int t = 0; t < 2; ++t) {
#pragma unroll
    for (int i = 0; i < 4; ++i) weight(t, t, i);
#pragma unroll
    for (int i = 0; i < B; ++i) row(t, t, i);
  }
  wait_requests<4 + B>();
  change();
  if (wa) change();  // the second group is one turn behind
  int pw = 0, px = 0;  // of stage t
  for (int t = 0; t < nk; ++t) {
    const int before = pw == 0 ? 2 : pw - 1;  // where stage t - 1 was
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int i = 0; i < 4; ++i) read_w(pw, 0, s, i);
#pragma unroll
      for (int j = 0; j < B; ++j) read_x(px, s, j);
      __builtin_amdgcn_sched_barrier(0);
      weight(t + 2, before, s);
      __builtin_amdgcn_sched_barrier(0);
    }
    wait_reads();
    change();
    products(0);
    change();
#pragma unroll
    for (int i = 0; i < 4 + (B > 2 ? B - 2 : 0); ++i) {
      if (i < 4) read_w(pw, 1, i / 2, i % 2 * 2), read_w(pw, 1, i / 2, i % 2 * 2 + 1);
      __builtin_amdgcn_sched_barrier(0);
      if (i < 2) weight(t + 2, before, 2 + i);
      else if (i - 2 < B) row(t + 2, px, i - 2);  // both groups have read them
      __builtin_amdgcn_sched_barrier(0);
    }
    wait_requests_and_reads<4 + B>();  // stage t + 1 has landed
    change();
    products(1);
    change();
    pw = pw == 2 ? 0 : pw + 1;
    px ^= 1;
  }
  if (!wa) change();
  wait_requests<0>();  // the repeated stages, before the LDS is given back
#pragma unroll
  for (int j = 0; j < B; ++j) {
    const int r = (wb * B + j) * 16 + r16;
    if (r >= nr) continue;
    const float s = p.scale ? p.wts[p.perm[lo + r]] : 1.f;
    bf16_t* y = reinterpret_cast<bf16_t*>(p.y) + (long long)(lo + r) * N;
#pragma unroll
    for (int h = 0; h < (UP ? 1 : 2); ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int n = n0 + wa * (UP ? 64 : 128) + h * 64 + i * 16 + 4 * g;
        if (n >= N) continue;  // (N % 4 == 0)
        float o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if constexpr (UP) {
            const float gt = acc[0][i][j][e] * s, up = acc[1][i][j][e] * s;
            o[e] = gt * __builtin_amdgcn_rcpf(1.f + __expf(-gt)) * up;
          } else {
            o[e] = acc[h][i][j][e] * s;
          }
        }
        *reinterpret_cast<uint2*>(y + n) = make_uint2(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]));
      }
  }
}

}  // namespace
