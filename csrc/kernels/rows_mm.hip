// y[M, N] = x[M, K] . W[N, K]^T (+ bias), bf16 or fp16, for the few rows of a short prompt.
#include "common.h"

namespace {

bool al16(const void* p) { return (uintptr_t)p % 16 == 0; }

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

constexpr int SK = 64, ROWS = 128;  // K a stage, activation rows at most

struct RowsPart {
  const void *x, *w, *bias;
  void* y;
  int N, K, act;  // act: 0 none, GELU 1 tanh, 2 erf
};
struct RowsArgs {
  // p[0], and beside it p[1] with blocks of its own (beside), or p[1]'s x and W along K: y[0] = x0 W0^T + x1 W1^T + both biases
  // (p[1].K without beside). p[1].K == 0: one product.
  RowsPart p[2];
  const void* res;  // two products along K: rows [M, N] that are added to their sums, or null
  float* ws;      // ks > 1: [block][slice][product tile][2][threads][2]
  unsigned* cnt;  // ks > 1: one arrival counter a block, zero before and after
  int M, ks, beside;
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t uniform_rsrc(const void* p) {
  const unsigned long long a = (unsigned long long)p;
  const unsigned long long u = ((unsigned long long)__builtin_amdgcn_readfirstlane((unsigned)(a >> 32)) << 32) |
                               (unsigned)__builtin_amdgcn_readfirstlane((unsigned)a);
  return __builtin_amdgcn_make_buffer_rsrc((void*)u, (short)0, -1, 0x00020000);
}

// both sub-steps' fragments of a stage and their wait in one piece (hipcc would drain every LDS-DMA in flight before a
// read it sees): runs of 16 rows at a0 and, for the second sub-step, at a1
__device__ __forceinline__ void read_frags(unsigned a0, unsigned a1, u32x4 (&r)[2][1]) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %3\n\ts_waitcnt lgkmcnt(0)"
               : "=&v"(r[0][0]), "=&v"(r[1][0])
               : "v"(a0), "v"(a1)
               : "memory");
#endif
}
__device__ __forceinline__ void read_frags(unsigned a0, unsigned a1, u32x4 (&r)[2][2]) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile(
      "ds_read_b128 %0, %4\n\tds_read_b128 %1, %4 offset:2048\n\t"
      "ds_read_b128 %2, %5\n\tds_read_b128 %3, %5 offset:2048\n\ts_waitcnt lgkmcnt(0)"
      : "=&v"(r[0][0]), "=&v"(r[0][1]), "=&v"(r[1][0]), "=&v"(r[1][1])
      : "v"(a0), "v"(a1)
      : "memory");
#endif
}
__device__ __forceinline__ void read_frags(unsigned a0, unsigned a1, u32x4 (&r)[2][4]) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile(
      "ds_read_b128 %0, %8\n\tds_read_b128 %1, %8 offset:2048\n\t"
      "ds_read_b128 %2, %8 offset:4096\n\tds_read_b128 %3, %8 offset:6144\n\t"
      "ds_read_b128 %4, %9\n\tds_read_b128 %5, %9 offset:2048\n\t"
      "ds_read_b128 %6, %9 offset:4096\n\tds_read_b128 %7, %9 offset:6144\n\ts_waitcnt lgkmcnt(0)"
      : "=&v"(r[0][0]), "=&v"(r[0][1]), "=&v"(r[0][2]), "=&v"(r[0][3]), "=&v"(r[1][0]), "=&v"(r[1][1]), "=&v"(r[1][2]),
        "=&v"(r[1][3])
      : "v"(a0), "v"(a1)
      : "memory");
#endif
}

// A block's first stage of its walk: neighbours at neighbouring ones, so that they find each other's activations in L2 (spread over all of K
// 128 rows of 4096 x 16384 40.5, 49.6 us), groups of 8 turned (16384 x 4096, a block a CU: 25.6; one after another 27.4)
__device__ __forceinline__ int walk_start(int blk, int stages) { return (blk ^ (blk >> 3)) % stages; }

template <bool F16>
__device__ __forceinline__ f32x4 mma(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (F16)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// Bound by the weight stream. A block is NB weight rows x all activation rows (rounded up to XR); a stage's weights and
// activations, 64 of K each, go straight to LDS (no registers), 64 to 96 KiB a workgroup;
// the products (weights as the A operand: a lane holds one activation row and four outputs) hide under it. Blocks of 64 rows
// where they are no more than the CUs, or K is sliced: partial sums (4 bytes beside 2 of a weight, for every activation row) cost
// more than reading the activations once a block from L2 (61 rows of 16384 x 4096 25.4 us, of 4096 x 4096 12.9; blocks of 128 in twice
// the slices 29.2, 16.2; 64 in twice the slices, 32 rows of 4096 x 16384 and x 4096 30.2, 35.0). Where 64 rows make more blocks than CUs, 128 halve what the activations cost (`block_rows`).
// Blocks start their walks of K at different stages (`walk_start`): from the same one they read the same columns of all rows, 2K bytes
// apart, at one time, which few of the memory's channels hold. 61 rows, us, ordinary loads, from the first stage and this: 12288 x 4096 26.3, 24.3;
// 16384 x 4096 32.1, 25.6; 4096 x 16384 34.3, 30.0; 14336 x 14336 93.1, 86.0; loads alone of 16384 x 4096 30.2, 23.8. Weights packed so that a
// stage is one piece of memory come to the same (24.4). The order of the sums follows from the block, the same at every run.
// Where the blocks are fewer than the CUs, slices of K write partial sums and the last to arrive adds them in slice order.
// An LDS-DMA instruction fills 8 rows of 128 bytes lane by lane, so the 16-byte pieces are swizzled (by row pair: 16 rows x one
// piece cover all 64 banks) on the source address.
// us, hipBLASLt : this (weights cold, both in a captured graph; at the copy rate 20.9, 27.8, 7.0, 27.8, 86):
//   rows   12288 x 4096   16384 x 4096   4096 x 4096   4096 x 16384   50400 x 4096
//     16    28.1 : 19.4    33.1 : 23.2   15.3 : 11.0   30.1 : 25.0    80.7 : 67.8
//     64    24.7 : 24.0    32.5 : 25.6   14.8 : 12.5   41.5 : 29.3    82.2 : 76.4
//    128    31.7 : 33.3    36.6 : 35.1   24.2 : 16.6   80.8 : 41.4    88.1 : 95.5
// Which sizes run here: few_rows in ops/linear.py.
// XR activation rows; W waves, WM of them across the activation rows (8 rather than 4 read less from LDS: 61 rows of 2048 x 8192 and x 2048
// 16.7, 15.9); SNB stages.
// TWO: another product beside this one, or more of K (RowsArgs).
template <bool F16, int NB, int W, int XR, int WM, int SNB, bool TWO>
__global__ void __launch_bounds__(64 * W, 2) rows_mm_kernel(RowsArgs p) {
  constexpr int WN = W / WM, A = NB / WN / 16, B = XR / WM / 16;  // a wave's runs of 16 weight and activation rows
  constexpr int XP = XR / 8, XI = (XP + W - 1) / W;  // pieces of 8 activation rows, requests a wave (7 waves: some of a piece that another one requests)
  constexpr int STG = (NB + XR) * SK * 2, WI = NB / 8 / W, PER = WI + XI;
  static_assert(WI * W * 8 == NB && A * WN * 16 == NB && B * WM * 16 == XR);
  extern __shared__ __attribute__((aligned(1024))) char sl[];  // [SNB][NB weight rows | XR activation rows][128 B]
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wn = wv % WN, wm = wv / WN;
  const int r16 = lane & 15, g = lane >> 4;
  const int id = xcd_remap(blockIdx.x, gridDim.x);  // the slices of a block on one XCD, beside their partial sums
  const int blk = id / p.ks, z = id % p.ks;
  const int nb0 = (p.p[0].N + NB - 1) / NB;
  const bool second = TWO && p.beside && blk >= nb0;
  const RowsPart q = second ? p.p[1] : p.p[0];
  const int n0 = (second ? blk - nb0 : blk) * NB;
  const int K2 = TWO && !p.beside ? p.p[1].K : 0;
  const int nka = q.K / SK, nk = nka + K2 / SK;
  const int t0 = (int)((long long)nk * z / p.ks), t1 = (int)((long long)nk * (z + 1) / p.ks);
  const __amdgpu_buffer_rsrc_t rw = uniform_rsrc(q.w), rx = uniform_rsrc(q.x);
  const __amdgpu_buffer_rsrc_t rw2 = uniform_rsrc(p.p[1].w), rx2 = uniform_rsrc(p.p[1].x);
  unsigned wo[WI], xo[XI], wo2[WI], xo2[XI];
  auto offsets = [&](int K, unsigned (&w)[WI], unsigned (&x)[XI]) {
#pragma unroll
    for (int i = 0; i < WI; ++i) {
      const int r = wv * 8 * WI + 8 * i + (lane >> 3);
      w[i] = ((unsigned)min(n0 + r, q.N - 1) * K + 8 * ((lane & 7) ^ ((r >> 1) & 7))) * 2;
    }
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      const int r = 8 * min(wv * XI + i, XP - 1) + (lane >> 3);
      x[i] = ((unsigned)min(r, p.M - 1) * K + 8 * ((lane & 7) ^ ((r >> 1) & 7))) * 2;
    }
  };
  offsets(q.K, wo, xo);
  if (TWO) offsets(K2, wo2, xo2);
  typedef __attribute__((address_space(3))) char lds_char;
  lds_char* lsm = (lds_char*)sl;
  const int first = t0 + walk_start(blk, t1 - t0);
  auto issue = [&](int t) {  // the walk's stage t: the last ones repeat one that nobody reads
    const int at = first + min(t, t1 - t0 - 1), tt = __builtin_amdgcn_readfirstlane(at < t1 ? at : at - (t1 - t0));
    lds_char* st = lsm + t % SNB * STG;
#if defined(__HIP_DEVICE_COMPILE__)
    const bool one = !TWO || tt < nka;
    const int k = (one ? tt : tt - nka) * SK * 2;
    const __amdgpu_buffer_rsrc_t fw = one ? rw : rw2, fx = one ? rx : rx2;
    // (the weights non-temporal: no other block reads them. 32 rows, cold, us: 12288 and 16384 x 4096 42.6, 37.8 (6.2 TB/s); 4096 x 16384 and x 4096
    // 34.7, 30.2; 50400 x 4096 82.8, 75.6; 61 rows 43.8, 40.1; 38.6, 37.2; 86.5, 81.7. Called over and over with nothing
    // else between, weights that the last cache (256 MB) would hold come slower, 180 MB of 2304 x 768 at 61 rows 6.2, 7.1, of 50304 x 768 16.1, 21.0; cold
    // they gain nothing below 2048 of width. But whole steps of models that small, which read a cache and logits too, are no faster with ordinary loads
    // of weights less than 2048 wide: GPT-J layers, 12 of 768 with their head, 16 rows of 100 tokens 404, 390; 64 506, 509; 128 of 200 703, 709; 8 of 1024 317,
    // 315; 386, 383; 594, 577; GPT-2's prompts of 16 to 120 tokens are bound by the host.)
#pragma unroll
    for (int i = 0; i < WI; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(fw, (void __attribute__((address_space(3)))*)(st + (wv * WI + i) * 1024), 16,
                                               one ? wo[i] : wo2[i], k, 0, 2);
#pragma unroll
    for (int i = 0; i < XI; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(fx, (void __attribute__((address_space(3)))*)(st + (NB / 8 + min(wv * XI + i, XP - 1)) * 1024), 16,
                                               one ? xo[i] : xo2[i], k, 0, 0);
#endif
  };
  f32x4 acc[A][B];
#pragma unroll
  for (int i = 0; i < A; ++i)
#pragma unroll
    for (int j = 0; j < B; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const unsigned base = (unsigned)(size_t)lsm, sw = (r16 >> 1) & 7;
  const unsigned aw = (wn * A * 16 + r16) * 128, ax = (NB + wm * B * 16 + r16) * 128;
  const unsigned c0 = (g ^ sw) * 16, c1 = ((4 + g) ^ sw) * 16;
#pragma unroll
  for (int t = 0; t < SNB - 1; ++t) issue(t);
  for (int t = 0; t < t1 - t0; ++t) {
    // this wave's pieces of stage t have landed (SNB - 2 younger stages may be in flight), then everybody's
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((SNB - 2) * PER) : "memory");
    __builtin_amdgcn_s_barrier();
    issue(t + SNB - 1);  // into the buffer of stage t - 1, which all waves have left
    const unsigned st = base + t % SNB * STG;
    u32x4 wf[2][A], xf[2][B];
    read_frags(st + aw + c0, st + aw + c1, wf);
    read_frags(st + ax + c0, st + ax + c1, xf);
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int j = 0; j < B; ++j)
#pragma unroll
        for (int i = 0; i < A; ++i) acc[i][j] = mma<F16>(wf[s][i], xf[s][j], acc[i][j]);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the repeated stages, before the LDS is given back
  unsigned long long* const part = reinterpret_cast<unsigned long long*>(p.ws) + (long long)blk * p.ks * A * B * (128 * W) + threadIdx.x;
  if (p.ks > 1) {
#pragma unroll
    for (int i = 0; i < A; ++i)
#pragma unroll
      for (int j = 0; j < B; ++j)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          __hip_atomic_store(part + (z * A * B + i * B + j) * (128 * W) + h * (64 * W),
                             __builtin_bit_cast(unsigned long long, f32x2{acc[i][j][2 * h], acc[i][j][2 * h + 1]}),
                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
      const int last = __hip_atomic_fetch_add(p.cnt + blk, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)p.ks - 1;
      if (last) {
        __hip_atomic_store(p.cnt + blk, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      }
      *(int*)sl = last;  // (the stages are done)
    }
    __syncthreads();
    if (!*(volatile int*)sl) return;
  }
  uint2 res[A][B];  // requested before the other slices' sums
  if (TWO && p.res) {
#pragma unroll
    for (int i = 0; i < A; ++i)
#pragma unroll
      for (int j = 0; j < B; ++j) {
        const int n = min(n0 + (wn * A + i) * 16 + 4 * g, q.N - 4), m = min((wm * B + j) * 16 + r16, p.M - 1);
        res[i][j] = *reinterpret_cast<const uint2*>(reinterpret_cast<const unsigned short*>(p.res) + (long long)m * q.N + n);
      }
  }
  if (p.ks > 1) {
    // all slices in slice order, whichever came last: the sum does not depend on the order of arrival
    f32x4 sum[A][B];
#pragma unroll
    for (int i = 0; i < A; ++i)
#pragma unroll
      for (int j = 0; j < B; ++j) sum[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
    for (int s = 0; s < p.ks; ++s) {
#pragma unroll
      for (int i = 0; i < A; ++i)
#pragma unroll
        for (int j = 0; j < B; ++j) {
          const auto* q = part + (s * A * B + i * B + j) * (128 * W);
          const f32x2 lo = __builtin_bit_cast(f32x2, q[0]), hi = __builtin_bit_cast(f32x2, q[64 * W]);
          sum[i][j] += f32x4{lo[0], lo[1], hi[0], hi[1]};
        }
    }
#pragma unroll
    for (int i = 0; i < A; ++i)
#pragma unroll
      for (int j = 0; j < B; ++j) acc[i][j] = sum[i][j];
  }
#pragma unroll
  for (int i = 0; i < A; ++i) {
    const int n = n0 + (wn * A + i) * 16 + 4 * g;
    if (n >= q.N) continue;
    float b[4] = {0.f, 0.f, 0.f, 0.f};
    auto add_bias = [&](const void* bias) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const unsigned short v = reinterpret_cast<const unsigned short*>(bias)[n + e];
        b[e] += F16 ? (float)__builtin_bit_cast(_Float16, v) : bf2f(v);
      }
    };
    if (q.bias) add_bias(q.bias);
    if (TWO && K2 && p.p[1].bias) add_bias(p.p[1].bias);
#pragma unroll
    for (int j = 0; j < B; ++j) {
      const int m = (wm * B + j) * 16 + r16;
      if (m >= p.M) continue;
      float o[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        o[e] = acc[i][j][e] + b[e];
        if (q.act) o[e] = q.act == 1 ? gelu_tanh(o[e]) : gelu_erf(o[e]);
      }
      if (TWO && p.res) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const unsigned short v = (e < 2 ? res[i][j].x : res[i][j].y) >> 16 * (e & 1);
          o[e] += F16 ? (float)__builtin_bit_cast(_Float16, v) : bf2f(v);
        }
      }
      uint2 v;
      if constexpr (F16) {
        const _Float16 h[4] = {(_Float16)o[0], (_Float16)o[1], (_Float16)o[2], (_Float16)o[3]};
        v = __builtin_bit_cast(uint2, h);
      } else {
        v = make_uint2(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]));
      }
      *reinterpret_cast<uint2*>(reinterpret_cast<unsigned short*>(q.y) + (long long)m * q.N + n) = v;
    }
  }
}

int blocks_of(const RowsArgs& a, int nb) { return (a.p[0].N + nb - 1) / nb + (a.beside ? (a.p[1].N + nb - 1) / nb : 0); }

template <bool F16, int NB, int W, int XR, int WM, int SNB, bool TWO>
int go_as(const RowsArgs& a, hipStream_t s) {
  constexpr int lds = SNB * (NB + XR) * SK * 2;
  if (hipFuncSetAttribute((const void*)rows_mm_kernel<F16, NB, W, XR, WM, SNB, TWO>, hipFuncAttributeMaxDynamicSharedMemorySize, lds) !=
      hipSuccess)
    return 5;
  hipLaunchKernelGGL((rows_mm_kernel<F16, NB, W, XR, WM, SNB, TWO>), dim3(blocks_of(a, NB) * a.ks), dim3(64 * W), lds, s, a);
  return hipGetLastError() == hipSuccess ? 0 : 4;
}
template <bool F16, int NB, int W, int XR, int WM, int SNB>
int go(const RowsArgs& a, hipStream_t s) {
  return a.p[1].K ? go_as<F16, NB, W, XR, WM, SNB, true>(a, s) : go_as<F16, NB, W, XR, WM, SNB, false>(a, s);
}

// Blocks of 128 weight rows: where 64 make more blocks than CUs and 128 fill whole rounds of them better. us, 61 rows, 64 and 128 a block
// (x 4096): 18432 44.0, 35.2; 24576 46.9, 37.7; 12288 and 16384 beside each other 51, 41.7; 32768 48.9, 46.1; 50400 93, 80.6; 57344 99.5, 88.6; a
// second round of a few blocks loses: 36864 70.5, 73.9; 43008 71.9, 77.1; not for 128 rows, whose products cost as much as their weights: 91.8, 88.6.
// Blocks of 112, two a CU, where its most loaded CU has fewer rows then: 32 rows, 128 and 112 a block: 50400 x 4096 75.1, 71.0, x 2048 41.4, 37.0; 57344 78.9,
// 75.3, 42.1, 39.5; one round of blocks gains nothing (28672 x 4096, 224 blocks and 256, 39.3, 40.0).
int block_rows(const RowsArgs& a, int xr) {
  if (a.ks > 1 || blocks_of(a, 64) <= 256) return 64;
  const int n = blocks_of(a, 128), rounds = (n + 255) / 256;
  if (xr == 128 || n <= 256) return 128;
  if (n <= 384) return 64;
  return (blocks_of(a, 112) + 255) / 256 * 112 < rounds * 128 ? 112 : 128;
}

// Checks what the kernel asks of its arguments and launches it
int rows_mm(int dtype, const RowsArgs& a, long long ws_floats, int cnt_n, hipStream_t s) {
  if ((dtype != 1 && dtype != 2) || a.M < 1 || a.M > ROWS || a.ks < 1) return 1;
  const int parts = a.p[1].K ? 2 : 1;
  long long blocks = 0, stages = 0;
  for (int i = 0; i < parts; ++i) {
    const RowsPart& q = a.p[i];
    const bool out = i == 0 || a.beside;  // has rows of its own
    if (!q.x || !q.w || (out && !q.y) || q.N < 16 || q.N % 16 || q.K < SK || q.K % SK || q.act < 0 || q.act > 2) return 1;
    if (!out && q.N != a.p[0].N) return 1;
    if (a.beside && a.ks > q.K / SK) return 1;
    if (!al16(q.x) || !al16(q.w) || (out && (uintptr_t)q.y % 8)) return 2;
    if (2ll * (q.N > a.M ? q.N : a.M) * q.K >= 1ll << 32) return 3;  // (32-bit byte offsets into W and x)
    if (out) blocks += (q.N + 63) / 64;
    stages += q.K / SK;
  }
  if (!a.beside && a.ks > stages) return 1;
  const int xr = a.M <= 32 ? 32 : a.M <= 64 ? 64 : 128;
  if (blocks * a.ks >= 1ll << 31) return 3;
  if (a.ks > 1 && (!a.ws || !a.cnt || !al16(a.ws) || ws_floats < blocks * a.ks * 64 * xr || cnt_n < blocks)) return 6;
  const bool f16 = dtype == 2;
  const int nb = block_rows(a, xr);
  if (nb == 112) {
    if (xr == 32) return f16 ? go<true, 112, 7, 32, 1, 4>(a, s) : go<false, 112, 7, 32, 1, 4>(a, s);
    return f16 ? go<true, 112, 7, 64, 1, 3>(a, s) : go<false, 112, 7, 64, 1, 3>(a, s);
  }
  if (nb == 128) {
    if (xr == 32) return f16 ? go<true, 128, 4, 32, 1, 4>(a, s) : go<false, 128, 4, 32, 1, 4>(a, s);
    if (xr == 64) return f16 ? go<true, 128, 8, 64, 2, 4>(a, s) : go<false, 128, 8, 64, 2, 4>(a, s);
    return f16 ? go<true, 128, 8, 128, 2, 3>(a, s) : go<false, 128, 8, 128, 2, 3>(a, s);
  }
  if (xr == 32) return f16 ? go<true, 64, 4, 32, 1, 6>(a, s) : go<false, 64, 4, 32, 1, 6>(a, s);
  if (xr == 64) return f16 ? go<true, 64, 8, 64, 2, 4>(a, s) : go<false, 64, 8, 64, 2, 4>(a, s);
  return f16 ? go<true, 64, 8, 128, 2, 3>(a, s) : go<false, 64, 8, 128, 2, 3>(a, s);
}

}  // namespace

// dtype 1 bf16, 2 fp16. x [M, K], W [N, K], y [M, N] contiguous, x and W 16-byte aligned; bias [N] or null; ks > 1: slices of
// K, with ws of ks * blocks * 64 * (M rounded up to 32, 64 or 128) floats and cnt of `blocks` zeroed counters (left zeroed),
// blocks = ceil(N / 64). Other sizes return a status and launch nothing.
KCA_API int kca_rows_mm(int dtype, const void* x, const void* w, const void* bias, void* y, float* ws, unsigned* cnt,
                        long long ws_floats, int cnt_n, int M, int N, int K, int ks, hipStream_t s) {
  return rows_mm(dtype, RowsArgs{{{x, w, bias, y, N, K, 0}, {}}, nullptr, ws, cnt, M, ks, 0}, ws_floats, cnt_n, s);
}

// One product with a GELU (act: 0 none, 1 tanh, 2 erf) on its fp32 sums (x2 null), or two: beside each other, y2 [M, N2] =
// act2(x2 W2^T + bias2) in blocks of its own, or (beside 0) along K: y = act(x W^T + x2 W2^T + bias + bias2), N2 == N. Blocks: both
// products' where they lie beside each other. res (along K, no act): rows [M, N] of y's type, 8-byte aligned, added to the fp32 sums; or null.
KCA_API int kca_rows_mm_two(int dtype, int beside, const void* x, const void* w, const void* bias, void* y, int N, int K, int act,
                            const void* x2, const void* w2, const void* bias2, void* y2, int N2, int K2, int act2,
                            const void* res, float* ws, unsigned* cnt, long long ws_floats, int cnt_n, int M, int ks, hipStream_t s) {
  if ((x2 && K2 < SK) || (res && (!x2 || beside || act))) return 1;
  if ((uintptr_t)res % 8) return 2;
  return rows_mm(dtype, RowsArgs{{{x, w, bias, y, N, K, act}, {x2, w2, bias2, y2, N2, x2 ? K2 : 0, act2}}, res, ws, cnt, M, ks, x2 && beside},
                 ws_floats, cnt_n, s);
}
