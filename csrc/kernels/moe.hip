// Mixture of gated experts: router, grouping, expert products.
//
//   s = sigmoid(W_router h); the `top` experts with the largest scores take the token, with weight s;  or
//   s = softmax(W_router h); the `top` experts with the largest s + correction, out of the `keep` of `groups` equal groups
//   of neighbours whose largest such score is largest, with weight s / (their sum + 1e-20). The last `identity` of the
//   outputs have no weights: they pass the token on (norm_residual.hip adds it), and no expert row is made for them.
//   expert(x) = W_down (silu(W_gate x) * (W_up x))
// A weight scales the expert's input -- both first products are linear, so it multiplies their fp32 sums
// before the activation -- or its output (`scale_in` 0). The router (and the shared expert's gate, one
// more row) accumulates in fp32 and is never rounded.
//
//   route   scores, top-k, weights of each token (bf16: matrix cores, 16 tokens per workgroup)
//   group   assignments sorted by expert and cut in row tiles that hold one expert each
//   gemv    expert products of tiles of up to 8 rows: streams the weight rows on the vector units
//           (decode; any dims, fp32 too)
//   stream  expert products of tiles of up to 32 rows on the matrix cores (large decode batches, short prompts)
//   gemm    expert products of tiles of up to 256 rows on the matrix cores (prompts)
// Expert weights are stacked: gate-and-up [E][2F][d] (gate rows first), down [E][d][F]. The sorted rows'
// activations are [n][F], their outputs [n][d]; the residual pass (rms_shift.hip) sums a token's outputs
// through `inv`.
#include "common.h"
#include "expert_tiles.h"
#include "lanes.h"

#include <type_traits>

namespace {

template <typename E> __device__ __forceinline__ float lde(const E* p);
template <> __device__ __forceinline__ float lde<float>(const float* p) { return *p; }
template <> __device__ __forceinline__ float lde<bf16_t>(const bf16_t* p) { return bf2f(*p); }
template <typename E> __device__ __forceinline__ void ste(E* p, float v);
template <> __device__ __forceinline__ void ste<float>(float* p, float v) { *p = v; }
template <> __device__ __forceinline__ void ste<bf16_t>(bf16_t* p, float v) { *p = f2bf(v); }

__device__ __forceinline__ float sigmoid(float x) { return 1.f / (1.f + expf(-x)); }

struct RouteArgs {
  const void* h;       // [T][d]
  const void* wr;      // [E][d]
  const void* wsg;     // [d] shared expert's gate (nullable)
  int* ids;            // [T][top]
  float* wts;          // [T][top]
  float* sg;           // [T]
  int T, d, E, top;    // E: router outputs, identity experts included
  int softmax, groups, keep;
  const float* fix;    // [E] correction of the choice (softmax; nullable)
};

__device__ __forceinline__ void lds_order() {  // one wave's LDS writes before its later reads
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// largest of z[0 .. n) over the wave; ties go to the lower index
__device__ __forceinline__ void wave_argmax(const float* z, int n, int lane, float& best, int& bi) {
  best = -INFINITY;
  bi = 0x7fffffff;
  for (int e = lane; e < n; e += 64)
    if (z[e] > best) best = z[e], bi = e;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float ob = __shfl_xor(best, o, 64);
    const int oi = __shfl_xor(bi, o, 64);
    if (ob > best || (ob == best && oi < bi)) best = ob, bi = oi;
  }
  if (bi >= n) bi = 0;  // (no finite score left)
}

// One wave: softmax scores, corrected choice within the best groups. z: logits, c, w: E floats each (LDS).
__device__ __forceinline__ void pick_softmax(const RouteArgs& p, float* z, float* c, float* w, int t, int lane, int* ids_lds) {
  float mx = -INFINITY, sum = 0.f;
  for (int e = lane; e < p.E; e += 64) mx = fmaxf(mx, z[e]);
  mx = wave_max(mx);
  for (int e = lane; e < p.E; e += 64) sum += expf(z[e] - mx);
  sum = 1.f / wave_sum(sum);
  for (int e = lane; e < p.E; e += 64) {
    const float s = expf(z[e] - mx) * sum;
    z[e] = s;
    c[e] = s + (p.fix ? p.fix[e] : 0.f);
  }
  lds_order();
  if (p.keep < p.groups) {
    const int size = p.E / p.groups;
    for (int g = lane; g < p.groups; g += 64) {
      float best = -INFINITY;
      for (int e = g * size; e < (g + 1) * size; ++e) best = fmaxf(best, c[e]);
      w[g] = best;
    }
    lds_order();
    for (int g = lane; g < p.groups; g += 64) {
      int ahead = 0;  // groups before this one
      for (int j = 0; j < p.groups; ++j) ahead += w[j] > w[g] || (w[j] == w[g] && j < g);
      if (ahead >= p.keep)
        for (int e = g * size; e < (g + 1) * size; ++e) c[e] = -INFINITY;
    }
    lds_order();
  }
  float total = 0.f;
  for (int k = 0; k < p.top; ++k) {
    float best;
    int bi;
    wave_argmax(c, p.E, lane, best, bi);
    total += z[bi];
    if (lane == 0) {
      p.ids[(long long)t * p.top + k] = bi;
      if (ids_lds) ids_lds[t * p.top + k] = bi;
      w[k] = z[bi];
      c[bi] = -INFINITY;
    }
    lds_order();
  }
  for (int k = lane; k < p.top; k += 64) p.wts[(long long)t * p.top + k] = w[k] / (total + 1e-20f);
}

__device__ __forceinline__ float lane_of(float v, int j) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), j));
}

// largest over the wave, in every lane (rows of 16 by DPP, the four rows by lane reads)
__device__ __forceinline__ float lanes_max(float x) {
  x = lanes_reduce<16>(x, [](float a, float b) { return fmaxf(a, b); });
  return fmaxf(fmaxf(lane_of(x, 0), lane_of(x, 16)), fmaxf(lane_of(x, 32), lane_of(x, 48)));
}

// Both rules for up to 64 outputs, one a lane. (NaN counts as the least; ties go to the lower index.) The largest is
// taken `top` times, or, where that is more than half of the outputs, all ranks are counted at once: 16 instructions a
// choice, 8 an output (1 token, top 2 of 16, one workgroup: counting 11.7 us, taking 8.9).
__device__ __forceinline__ void pick_lanes(const RouteArgs& p, const float* z, float fix, int t, int lane, int* ids_lds) {
  const bool on = lane < p.E;
  float s = on ? z[lane] : -INFINITY, c;
  if (p.softmax) {
    auto add = [](float a, float b) { return a + b; };
    const float mx = lanes_max(s), e = on ? expf(s - mx) : 0.f;
    s = e / lanes_reduce<64>(e, add);
    c = on ? s + fix : -INFINITY;
    if (c != c) c = -INFINITY;
    if (p.keep < p.groups) {
      const int size = p.E / p.groups, g = lane / size;
      auto big = [](float a, float b) { return fmaxf(a, b); };
      float best = c;
      if (size == 8) best = lanes_reduce<8>(c, big);
      else if (size == 16) best = lanes_reduce<16>(c, big);
      else if (size == 4) best = lanes_reduce<4>(c, big);
      else
        for (int j = 0; j < size; ++j) best = fmaxf(best, __shfl(c, g * size + j, 64));
      int ahead = 0;  // groups before this lane's
      for (int j = 0; j < p.groups; ++j) {
        const float o = lane_of(best, j * size);
        ahead += o > best || (o == best && j < g);
      }
      if (ahead >= p.keep) c = -INFINITY;
    }
  } else {
    c = s != s ? -INFINITY : s;
  }
  int rank = 64;
  if (2 * p.top <= p.E) {
    unsigned long long left = p.E == 64 ? ~0ull : (1ull << p.E) - 1;
    float m = on ? c : -INFINITY;
    for (int k = 0; k < p.top; ++k) {
      const float best = lanes_max(m);
      const int at = __builtin_ctzll(__ballot(c == best) & left);
      left &= ~(1ull << at);
      if (lane == at) rank = k, m = -INFINITY;
    }
  } else {
    rank = 0;
    for (int j = 0; j < p.E; ++j) {
      const float o = lane_of(c, j);
      rank += o > c || (o == c && j < lane);
    }
  }
  const bool take = on && rank < p.top;
  float w = sigmoid(s);
  if (p.softmax) w = s / (lanes_reduce<64>(take ? s : 0.f, [](float a, float b) { return a + b; }) + 1e-20f);
  if (take) {
    // (written through: route_split_kernel's last workgroup reads what others chose)
    __hip_atomic_store(p.ids + (long long)t * p.top + rank, lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (ids_lds) ids_lds[t * p.top + rank] = lane;
    p.wts[(long long)t * p.top + rank] = w;
  }
}

// this lane's correction, requested early
__device__ __forceinline__ float lane_fix(const RouteArgs& p, int lane) { return p.fix && p.E <= 64 && lane < p.E ? p.fix[lane] : 0.f; }

// One wave: the top experts of one token from its logits z[E] (LDS; softmax: E floats each at c and w).
__device__ __forceinline__ void pick(const RouteArgs& p, float* z, float* c, float* w, float fix, int t, int lane, int* ids_lds = nullptr) {
  if (p.E <= 64) return pick_lanes(p, z, fix, t, lane, ids_lds);
  if (p.softmax) return pick_softmax(p, z, c, w, t, lane, ids_lds);
  for (int k = 0; k < p.top; ++k) {
    float best;
    int bi;
    wave_argmax(z, p.E, lane, best, bi);
    if (lane == 0) {
      p.ids[(long long)t * p.top + k] = bi;
      if (ids_lds) ids_lds[t * p.top + k] = bi;
      p.wts[(long long)t * p.top + k] = sigmoid(best);
      z[bi] = -INFINITY;
    }
    lds_order();
  }
}

// any dims and type: one token per workgroup, a wave per expert row
template <typename E>
__global__ void __launch_bounds__(256) route_rows_kernel(RouteArgs p) {
  extern __shared__ float z[];  // [E + 1], softmax: [2][E] more
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, t = blockIdx.x;
  const E* h = reinterpret_cast<const E*>(p.h) + (long long)t * p.d;
  const int n = p.E + (p.wsg ? 1 : 0);
  for (int e = wv; e < n; e += 4) {
    const E* w = e < p.E ? reinterpret_cast<const E*>(p.wr) + (long long)e * p.d : reinterpret_cast<const E*>(p.wsg);
    float s = 0.f;
    for (int i = lane; i < p.d; i += 64) s = fmaf(lde<E>(h + i), lde<E>(w + i), s);
    s = wave_sum(s);
    if (lane == 0) z[e] = s;
  }
  __syncthreads();
  if (wv == 0) pick(p, z, z + n, z + n + p.E, lane_fix(p, lane), t, lane);
  if (threadIdx.x == 64 && p.wsg) p.sg[t] = sigmoid(z[p.E]);
}

struct GroupArgs {
  const int* ids;      // [n]; E and beyond: no expert row (inv -1)
  int n, E, mt;
  int *perm, *inv, *tiles, *ntiles;
};

// Tiles of up to 256 rows: an expert's rows in units of 64 (a product's steps), as evenly over its tiles as they go: `more` tiles of
// per + 1 units, then the others. (Full tiles and a short last one, whose weights then came from memory once more: sublayer of 4096
// tokens, 16 experts of 3 x 4096 x 4096, top 2 893 us, evenly 850.) Experts stand by their largest tile: expert_turns_kernel.
struct Cut {
  int tiles, per, more;
};
__device__ __forceinline__ Cut cut(int c) {
  const int u = (c + 63) / 64, nt = (u + 3) / 4;
  return nt ? Cut{nt, u / nt, u % nt} : Cut{0, 0, 0};
}

// n assignments -> perm (sorted position -> assignment), inv (assignment -> sorted position), tiles
// [ntiles][5] (expert, first sorted position, rows <= mt, first tile and tile count of the expert) and
// their count. Late tiles stand after all others, each by itself, so that a product takes them last (expert_gemm_kernel); where the limit
// is 256 (BY_SIZE) the largest tiles stand first. One workgroup of NT threads; sh: 4 E + 3 ints.
template <int NT, bool BY_SIZE>
__device__ __forceinline__ void group_as(const GroupArgs& p, int* sh) {
  const int E = p.E, n = p.n, mt = p.mt, tid = threadIdx.x;
  int *cnt = sh, *off = sh + E, *toff = off + E + 1, *soff = toff + E + 1;
  constexpr int R = 4;  // a thread's first ids, read once for both passes
  int first[R];
#pragma unroll
  for (int j = 0; j < R; ++j) first[j] = p.ids[min(tid + j * NT, n - 1)];
  auto each = [&](auto&& f) {
#pragma unroll
    for (int j = 0; j < R; ++j)
      if (tid + j * NT < n) f(tid + j * NT, first[j]);
    for (int i = tid + R * NT; i < n; i += NT) f(i, p.ids[i]);
  };
  for (int e = tid; e < E; e += NT) cnt[e] = 0;
  __syncthreads();
  each([&](int, int e) {
    if (e < E) atomicAdd(&cnt[e], 1);
  });
  __syncthreads();
  if (tid < 64) {  // exclusive sums over the experts, 64 at a time
    int co = 0, so = 0;
    unsigned to = 0, to2 = 0;  // BY_SIZE: four sums in 16 bits each (group_rows: no more tiles), of experts whose largest tile is 4 .. 1 units
    for (int e0 = 0; e0 < E; e0 += 64) {
      const int e = e0 + tid, c = e < E ? cnt[e] : 0, small = late_tile(c, mt);
      const unsigned before2 = to2;
      int cs = c, b = 0;
      unsigned t = (c + mt - 1) / mt - small, t2 = 0;
      if constexpr (BY_SIZE) {
        const Cut k = cut(c);
        b = 4 - k.per - (k.more > 0);
        t = b < 2 ? k.tiles << 16 * b : 0, t2 = b < 2 ? 0 : k.tiles << 16 * (b & 1);
      }
      unsigned ts = t, ts2 = t2;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int a = __shfl_up(cs, o, 64);
        const unsigned b1 = __shfl_up(ts, o, 64);
        if (tid >= o) cs += a, ts += b1;
      }
      if constexpr (BY_SIZE) {
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
          const unsigned b2 = __shfl_up(ts2, o, 64);
          if (tid >= o) ts2 += b2;
        }
        to2 += __shfl(ts2, 63, 64);
      }
      const unsigned long long m = __ballot(small);
      if (e < E) {
        const unsigned u = to + ts - t, u2 = before2 + ts2 - t2;
        off[e] = co + cs - c;
        toff[e] = BY_SIZE ? (b < 2 ? u : u2) >> 16 * (b & 1) & 0xffff : u;
        soff[e] = BY_SIZE ? b : so + __popcll(m & ((1ull << tid) - 1));
      }
      co += __shfl(cs, 63, 64);
      to += __shfl(ts, 63, 64);
      so += __popcll(m);
    }
    if constexpr (BY_SIZE) {  // largest tiles first
      const unsigned n0 = to & 0xffff, n1 = n0 + (to >> 16), n2 = n1 + (to2 & 0xffff);
      for (int e = tid; e < E; e += 64) toff[e] += soff[e] == 0 ? 0 : soff[e] == 1 ? n0 : soff[e] == 2 ? n1 : n2;
      to = n2 + (to2 >> 16);
    }
    if (tid == 0) off[E] = co, toff[E] = to, *p.ntiles = to + so;
  }
  __syncthreads();
  for (int e = tid; e < E; e += NT) {
    const int c = cnt[e], nt = (c + mt - 1) / mt, small = late_tile(c, mt);
    const Cut k = BY_SIZE ? cut(c) : Cut{0, 0, 0};
    for (int j = 0; j < nt; ++j) {
      const bool last = small && j == nt - 1;  // (it stands alone)
      const int at = last ? toff[E] + soff[e] : toff[e] + j;
      const int from = BY_SIZE ? 64 * (j * k.per + min(j, k.more)) : j * mt;
      const int to = min(c, BY_SIZE ? from + 64 * (k.per + (j < k.more)) : from + mt);
      int* t = p.tiles + at * 5;
      t[0] = e;
      t[1] = off[e] + from;
      t[2] = to - from;
      t[3] = last ? at : toff[e];
      t[4] = last ? 1 : nt - small;
    }
    cnt[e] = off[e];
  }
  __syncthreads();
  each([&](int i, int e) {  // (the order within an expert does not matter: rows are independent)
    const int pos = e < E ? atomicAdd(&cnt[e], 1) : -1;
    if (pos >= 0) p.perm[pos] = i;
    p.inv[i] = pos;
  });
}

// (the second scan would cost other limits 0.8 us, its branches 0.25. Past 65535 tiles a class's count would not fit its 16 bits: in order of
// the experts then, full tiles and a rest)
template <int NT>
__device__ __forceinline__ void group_rows(const GroupArgs& p, int* sh) {
  if (p.mt == 256 && min(p.E, p.n) + p.n / 256 <= 0xffff) group_as<NT, true>(p, sh);
  else group_as<NT, false>(p, sh);
}

__global__ void __launch_bounds__(1024) group_kernel(GroupArgs p) {
  extern __shared__ int sh[];
  group_rows<1024>(p, sh);
}

// bf16: 16 tokens per workgroup, the K range cut over NW waves, 64 experts at a time. GROUP: the launch is
// one workgroup, which also groups its assignments (the decode step)
template <int NW, bool GROUP>
__global__ void __launch_bounds__(NW * 64) route_mfma_kernel(RouteArgs p, GroupArgs gr) {
  // z[16][zs], softmax: two more of them; part[NW][16][64] (then group_rows'), ids
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int n = p.E + (p.wsg ? 1 : 0), zs = (n + 63) / 64 * 64, zr = 16 * zs;
  float *z = lds, *part = lds + (p.softmax ? 3 : 1) * zr;
  int* sids = reinterpret_cast<int*>(part + NW * 1024);  // GROUP: [T * top]
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, r16 = lane & 15, g = lane >> 4;
  const int t0 = blockIdx.x * 16, d = p.d;
  const bf16_t* h = reinterpret_cast<const bf16_t*>(p.h) + (long long)min(t0 + r16, p.T - 1) * d;
  const int nk = (d + 31) / 32;
  const float fix = lane_fix(p, lane);
  for (int e0 = 0; e0 < n; e0 += 64) {
    const bf16_t* w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int e = min(e0 + 16 * i + r16, n - 1);
      w[i] = e < p.E ? reinterpret_cast<const bf16_t*>(p.wr) + (long long)e * d : reinterpret_cast<const bf16_t*>(p.wsg);
    }
    const int nt = min(4, (n - e0 + 15) / 16);
    f32x4 acc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto steps = [&](auto ntc) {
      constexpr int NTC = decltype(ntc)::value, AH = NTC > 2 ? 4 : 8;  // k steps whose loads fly together
      for (int k0 = wv * 2; k0 < nk; k0 += NW * AH) {  // 64 columns at a time: whole cache lines of every row
        u32x4 a[AH][NTC], b[AH];
#pragma unroll
        for (int j = 0; j < AH; ++j) {  // (no load is conditional; columns past d multiply zeros)
          const int c = (k0 + (j & 1) + (j >> 1) * NW * 2) * 32 + g * 8, cc = min(c, d - 8);
          const uint32_t keep = c < d ? ~0u : 0u;
          b[j] = *reinterpret_cast<const u32x4*>(h + cc) & u32x4{keep, keep, keep, keep};
#pragma unroll
          for (int i = 0; i < NTC; ++i) a[j][i] = *reinterpret_cast<const u32x4*>(w[i] + cc);
        }
        asm volatile("" ::: "memory");
#pragma unroll
        for (int j = 0; j < AH; ++j)
#pragma unroll
          for (int i = 0; i < NTC; ++i)
            acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[j][i]), __builtin_bit_cast(bf16x8, b[j]),
                                                             acc[i], 0, 0, 0);
      }
    };
    if (nt == 1) steps(std::integral_constant<int, 1>{});
    else if (nt == 2) steps(std::integral_constant<int, 2>{});
    else steps(std::integral_constant<int, 4>{});
    __syncthreads();
    // (16-byte pieces swizzled by row: 16 rows x one piece cover all 64 banks)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i < nt) *reinterpret_cast<f32x4*>(part + (wv * 16 + r16) * 64 + (((i * 4 + g) ^ r16) << 2)) = acc[i];
    __syncthreads();
    for (int i = tid; i < 256; i += NW * 64) {  // (row, piece)
      const int r = i >> 4, q = i & 15;
      if (q >= nt * 4) continue;
      f32x4 s{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w8 = 0; w8 < NW; ++w8) s += *reinterpret_cast<const f32x4*>(part + (w8 * 16 + r) * 64 + ((q ^ r) << 2));
      *reinterpret_cast<f32x4*>(z + r * zs + e0 + q * 4) = s;
    }
  }
  __syncthreads();
  for (int r = wv; r < 16; r += NW) {
    if (t0 + r >= p.T) break;
    if (p.wsg && lane == 0) p.sg[t0 + r] = sigmoid(z[r * zs + p.E]);
    pick(p, z + r * zs, z + zr + r * zs, z + 2 * zr + r * zs, fix, t0 + r, lane, GROUP ? sids : nullptr);
  }
  if constexpr (GROUP) {
    __syncthreads();
    gr.ids = sids;
    group_rows<NW * 64>(gr, reinterpret_cast<int*>(part));
  }
}

// bf16, up to 64 outputs and 1024 tokens: the 16 cuts of K that one workgroup of the kernel above takes, over four
// workgroups of four waves. Bound by a CU's loads: 16 token rows and 32 output rows of 2048 are 192 KiB, which one CU
// fetched in 11 us, its 16 waves' registers too few to request everything at once; a quarter of it is in flight whole.
// The last of the four adds the cuts (in the same order, so the logits are those of the kernel above, bit for bit),
// chooses and, GROUP, groups. parts: [token block][16 cuts][16 tokens][16 nt], cnt: a zeroed counter a token block.
// Sixteen waves although four of them load: one a token chooses (four tokens a wave, side by side, took twice as long).
// Routing and grouping, us, one workgroup a token block : this (launches back to back; 32 outputs of 2048, 16 of 4096, sigmoid):
//   1 token 12.4 : 7.2, 8.9 : 7.0; 16 tokens 15.9 : 8.2, 11.9 : 8.1; 128 tokens 17.6 : 10.2, 13.4 : 10.0;
//   1024 tokens 19.6 : 14.1, 14.5 : 13.0 (the blocks alone come near filling the chip)
// GROUP: 1, the launch is one token block, whose assignments it groups; 2, the last token block to be chosen groups all (cnt has one
// counter more), which took a launch of its own.
template <int GROUP>
__global__ void __launch_bounds__(1024) route_split_kernel(RouteArgs p, GroupArgs gr, float* parts, unsigned* cnt) {
  __shared__ __attribute__((aligned(16))) float z[16 * 64];
  __shared__ int sids[GROUP == 1 ? 16 * 64 : 1], sh[GROUP ? 4 * 64 + 3 : 1], s_last;
  const int n = p.E + (p.wsg ? 1 : 0), nt = (n + 15) / 16, d = p.d, nk = (d + 31) / 32;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, r16 = lane & 15, g = lane >> 4;
  const int tb = blockIdx.x / 4, cut = blockIdx.x % 4 * 4 + (wv & 3), t0 = tb * 16;
  const bf16_t* h = reinterpret_cast<const bf16_t*>(p.h) + (long long)min(t0 + r16, p.T - 1) * d;
  const float fix = lane_fix(p, lane);
  const bf16_t* w[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int e = min(16 * i + r16, n - 1);
    w[i] = e < p.E ? reinterpret_cast<const bf16_t*>(p.wr) + (long long)e * d : reinterpret_cast<const bf16_t*>(p.wsg);
  }
  f32x4 acc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto steps = [&](auto ntc, auto ahead) {
    constexpr int NTC = decltype(ntc)::value, AH = decltype(ahead)::value;
    for (int k0 = cut * 2; k0 < nk; k0 += 16 * AH) {  // 64 columns at a time: whole cache lines of every row
      u32x4 a[AH][NTC], b[AH];
#pragma unroll
      for (int j = 0; j < AH; ++j) {  // (no load is conditional; columns past d multiply zeros)
        const int c = (k0 + (j & 1) + (j >> 1) * 32) * 32 + g * 8, cc = min(c, d - 8);
        b[j] = *reinterpret_cast<const u32x4*>(h + cc);
#pragma unroll
        for (int i = 0; i < NTC; ++i) a[j][i] = *reinterpret_cast<const u32x4*>(w[i] + cc);
      }
      __builtin_amdgcn_sched_barrier(0);  // all requested before the first is waited for
#pragma unroll
      for (int j = 0; j < AH; ++j) {
        const int c = (k0 + (j & 1) + (j >> 1) * 32) * 32 + g * 8;
        const uint32_t keep = c < d ? ~0u : 0u;
        const u32x4 x = b[j] & u32x4{keep, keep, keep, keep};
#pragma unroll
        for (int i = 0; i < NTC; ++i)
          acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[j][i]), __builtin_bit_cast(bf16x8, x),
                                                           acc[i], 0, 0, 0);
      }
    }
  };
  auto store = [&] {
    auto* to = reinterpret_cast<unsigned long long*>(parts + ((long long)(tb * 16 + cut) * 16 + r16) * (16 * nt) + 4 * g);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i < nt) {
        const unsigned long long* v = reinterpret_cast<const unsigned long long*>(&acc[i]);
        __hip_atomic_store(to + 8 * i, v[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(to + 8 * i + 1, v[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
  };
  using std::integral_constant;
  if (wv < 4) {  // the other twelve waves choose
    const bool narrow = nk <= 64;  // four steps a cut
    if (nt == 1 && narrow) steps(integral_constant<int, 1>{}, integral_constant<int, 4>{});
    else if (nt == 1) steps(integral_constant<int, 1>{}, integral_constant<int, 8>{});
    else if (nt == 2 && narrow) steps(integral_constant<int, 2>{}, integral_constant<int, 4>{});
    else if (nt == 2) steps(integral_constant<int, 2>{}, integral_constant<int, 8>{});
    else steps(integral_constant<int, 4>{}, integral_constant<int, 4>{});
    store();
  }
  // The last of `of` workgroups to arrive at a zeroed counter, which it leaves zeroed, and which then reads what the others have
  // written through.
  auto last_of = [&](unsigned* c, unsigned of) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) {
      const int last = __hip_atomic_fetch_add(c, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == of - 1;
      if (last) {
        __hip_atomic_store(c, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      }
      s_last = last;
    }
    __syncthreads();
    return s_last != 0;
  };
  if (!last_of(cnt + tb, 4)) return;
  if (const int r = tid >> 4, q = tid & 15; r < 16 && q < nt * 4) {
    const float* from = parts + ((long long)tb * 256 + r) * (16 * nt) + 4 * q;
    f32x4 v[16], s{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < 16; ++c) v[c] = *reinterpret_cast<const f32x4*>(from + (long long)c * 256 * nt);
#pragma unroll
    for (int c = 0; c < 16; ++c) s += v[c];
    *reinterpret_cast<f32x4*>(z + r * 64 + 4 * q) = s;
  }
  __syncthreads();
  if (t0 + wv < p.T) {
    if (p.wsg && lane == 0) p.sg[t0 + wv] = sigmoid(z[wv * 64 + p.E]);
    pick_lanes(p, z + wv * 64, fix, t0 + wv, lane, GROUP == 1 ? sids : nullptr);
  }
  if constexpr (GROUP == 1) {
    __syncthreads();
    gr.ids = sids;
    group_rows<1024>(gr, sh);
  }
  if constexpr (GROUP == 2) {
    if (!last_of(cnt + gridDim.x / 4, gridDim.x / 4)) return;
    group_rows<1024>(gr, sh);
  }
}

// ------------------------------------------------------------------------------------------------ gemv
// Workgroup: one tile (<= MT rows of one expert, or of the shared one: the first tiles) x 4 waves, a wave streams two
// weight rows (gate and up of one output, or two outputs); the activation rows of a K chunk are staged in LDS for the four.
template <typename E, int MT, bool VEC>
__global__ void __launch_bounds__(256) expert_gemv_kernel(ExpertArgs p) {
  constexpr int KC = 2048, EPL = 16 / (int)sizeof(E), NL = KC / (64 * EPL);  // elements per lane and load
  extern __shared__ __attribute__((aligned(16))) char raw[];
  E* xs = reinterpret_cast<E*>(raw);  // [MT][KC]
  const int nsh = p.ws ? (p.tokens + MT - 1) / MT : 0;
  const bool sh = (int)blockIdx.y < nsh;
  const int tile = (int)blockIdx.y - nsh, N = sh ? p.Ns : p.N, K = sh ? p.Ks : p.K;
  if ((!sh && tile >= *p.ntiles) || (int)blockIdx.x * (p.up ? 4 : 8) >= N) return;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int* tl = p.tiles + (sh ? 0 : tile) * 5;
  const int ex = sh ? 0 : tl[0], lo = sh ? blockIdx.y * MT : tl[1], nr = sh ? min(MT, p.tokens - lo) : tl[2];
  const int n0 = p.up ? blockIdx.x * 4 + wv : (blockIdx.x * 4 + wv) * 2;
  const int rows = p.up ? 2 * N : N;
  const int ra = min(n0, N - 1), rb = p.up ? N + ra : min(n0 + 1, N - 1);
  const E* w = reinterpret_cast<const E*>(sh ? p.ws : p.w);
  const E* wa = w + ((long long)ex * rows + ra) * K;
  const E* wb = w + ((long long)ex * rows + rb) * K;
  float acc[2][MT];
#pragma unroll
  for (int r = 0; r < MT; ++r) acc[0][r] = acc[1][r] = 0.f;
  for (int k0 = 0; k0 < K; k0 += KC) {
    const int kn = min(KC, K - k0);
    u32x4 va[NL], vb[NL];
    if constexpr (VEC) {
#pragma unroll
      for (int i = 0; i < NL; ++i) {
        const int k = (i * 64 + lane) * EPL;
        if (k < kn) {
          va[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wa + k0 + k));
          vb[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wb + k0 + k));
        }
      }
    }
    __syncthreads();
    for (int r = 0; r < nr; ++r) {
      const long long src = p.up && !sh ? p.perm[lo + r] / p.top : lo + r;
      const E* x = reinterpret_cast<const E*>(sh ? p.xs : p.x) + src * K + k0;
      if constexpr (VEC) {
        for (int i = tid * EPL; i < kn; i += 256 * EPL)
          *reinterpret_cast<u32x4*>(xs + r * KC + i) = *reinterpret_cast<const u32x4*>(x + i);
      } else {
        for (int i = tid; i < kn; i += 256) xs[r * KC + i] = x[i];
      }
    }
    __syncthreads();
    if constexpr (VEC) {
#pragma unroll
      for (int i = 0; i < NL; ++i) {
        const int k = (i * 64 + lane) * EPL;
        if (k < kn) {
#pragma unroll
          for (int r = 0; r < MT; ++r)
            if (r < nr) {
              const u32x4 x = *reinterpret_cast<const u32x4*>(xs + r * KC + k);
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                if constexpr (sizeof(E) == 2) {
                  acc[0][r] = dot2_acc<0>(va[i][e], x[e], acc[0][r]);
                  acc[1][r] = dot2_acc<0>(vb[i][e], x[e], acc[1][r]);
                } else {
                  acc[0][r] = fmaf(__uint_as_float(va[i][e]), __uint_as_float(x[e]), acc[0][r]);
                  acc[1][r] = fmaf(__uint_as_float(vb[i][e]), __uint_as_float(x[e]), acc[1][r]);
                }
              }
            }
        }
      }
    } else {
      for (int k = lane; k < kn; k += 64) {
        const float a = lde<E>(wa + k0 + k), b = lde<E>(wb + k0 + k);
#pragma unroll
        for (int r = 0; r < MT; ++r)
          if (r < nr) {
            const float x = lde<E>(xs + r * KC + k);
            acc[0][r] = fmaf(a, x, acc[0][r]);
            acc[1][r] = fmaf(b, x, acc[1][r]);
          }
      }
    }
  }
#pragma unroll
  for (int r = 0; r < MT; ++r) {
    if (r >= nr) break;
    float a = wave_sum(acc[0][r]), b = wave_sum(acc[1][r]);
    if (lane) continue;
    if (p.scale && !sh) {
      const float s = p.wts[p.perm[lo + r]];
      a *= s;
      b *= s;
    }
    E* y = reinterpret_cast<E*>(sh ? p.ys : p.y) + (long long)(lo + r) * N;
    if (p.up) {
      if (n0 < N) ste<E>(y + n0, a * sigmoid(a) * b);
    } else {
      if (n0 < N) ste<E>(y + n0, a);
      if (n0 + 1 < N) ste<E>(y + n0 + 1, b);
    }
  }
}

// A launch's dimension holds less than 2^32 threads: more blocks stand in rows of 2^22 (a multiple of the 8 XCDs)
constexpr long long ROW_BLOCKS = 1 << 22;
dim3 block_rows(long long blocks) {
  return blocks <= ROW_BLOCKS ? dim3((unsigned)blocks) : dim3((unsigned)ROW_BLOCKS, (unsigned)((blocks + ROW_BLOCKS - 1) / ROW_BLOCKS));
}
__device__ __forceinline__ int block_number() { return blockIdx.y * (int)ROW_BLOCKS + blockIdx.x; }

template <typename F>
__device__ __forceinline__ void once_or_again(bool once, F&& f) {
  if (once) f(std::true_type{});
  else f(std::false_type{});
}

// ---------------------------------------------------------------------------------------------- stream
// (the tile: expert_tiles.h)
template <bool UP>
__global__ void __launch_bounds__(256, 2) expert_stream_kernel(ExpertArgs p) {
  extern __shared__ __attribute__((aligned(1024))) char sl[];
  constexpr int NB = UP ? SWN / 2 : SWN;
  const int nt = *p.ntiles, nb = (p.N + NB - 1) / NB;
  // Runs of 64 blocks, eight adjacent ones an XCD: what the chip reads at a time stays compact, and an expert's row tiles share an L2
  const int b = block_number(), end = nt * nb, c = b & ~63;
  if (b >= end) return;
  const int id = c + xcd_remap(b - c, min(64, end - c));
  const int* t0 = p.tiles + id / nb * 5;
  const int in = id - t0[3] * nb, tile = t0[3] + in % t0[4], bn = in / t0[4];
  const int* tl = p.tiles + tile * 5;
  const int nr = tl[2];
  once_or_again(read_once(tl[4], tl[2], p.mt), [&](auto once) {
    constexpr bool ONCE = decltype(once)::value;
    if (nr <= 8) expert_stream_tile<UP, 1, ONCE>(p, sl, tl[0], tl[1], nr, bn * NB);
    else if (nr <= 16) expert_stream_tile<UP, 2, ONCE>(p, sl, tl[0], tl[1], nr, bn * NB);
    else expert_stream_tile<UP, 4, ONCE>(p, sl, tl[0], tl[1], nr, bn * NB);
  });
}

template <bool UP>
__global__ void __launch_bounds__(256, 2) expert_block_kernel(ExpertArgs p) {
  extern __shared__ __attribute__((aligned(1024))) char sl[];
  constexpr int NB = UP ? BWN / 2 : BWN;
  const int nt = *p.ntiles, nb = (p.N + NB - 1) / NB, b = block_number();
  if (b >= nt * nb) return;
  const int id = xcd_remap(b, nt * nb);  // the order of expert_gemm_kernel
  const int* t0 = p.tiles + id / nb * 5;
  const int in = id - t0[3] * nb, tile = t0[3] + in % t0[4], bn = in / t0[4];
  const int* tl = p.tiles + tile * 5;
  once_or_again(read_once(tl[4], tl[2], p.mt), [&](auto once) { expert_block_tile<UP, decltype(once)::value>(p, sl, tl[0], tl[1], tl[2], bn * NB); });
}

// Whether a product of up to 32 rows a tile goes to blocks of 128 weight rows: past (K - 704) / 48 rows an expert, or, where blocks of 32 run all
// at one time, (K - 256) / 64; at most 30. One product, us, blocks of 32 weight rows and of 128 (outputs x K, experts):
//   down 1024 x 512, 64: 5 rows 15.4, 13.1; 16 rows 22.1, 18.2
//   down 2048 x 768, 24: 3 rows 15.7, 17.0; 5 rows 18.4, 18.4; 12 rows 21.6, 19.4; 20 rows 23.8, 19.1
//   down 2048 x 1024, 32: 5 rows 19.9, 20.8; 12 rows 28.2, 24.1; 26 rows 37.9, 34.3
//   up 512 x 1024, 16: 5 rows 9.2, 10.4; 12 rows 10.9, 11.3; 16 rows 13.5, 11.4; 26 rows 13.7, 11.1
//   up 704 x 1536, 32: 8 rows 25.6, 27.7; 16 rows 32.3, 31.5; 20 rows 35.1, 32.7
//   up 1024 x 2048, 32: 20 rows 57.9, 62.6; 26 rows 62.1, 61.7; 34 rows 67.8, 60.9    down 4096 x 4096, 8: 20 rows 57.4, 71.4; 34 rows 67.0, 67.2
static bool stream_block(int up, int N, int K, int top, int x_rows, int max_tiles) {
  const long long n = up ? (long long)x_rows * top : x_rows;
  const long long used = max_tiles - n / SROWS > 1 ? max_tiles - n / SROWS : 1;  // (max_tiles: experts and whole tiles)
  const bool once = used * ((N + (up ? SWN / 2 : SWN) - 1) / (up ? SWN / 2 : SWN)) <= 512;
  return n > 30 * used || (once ? 64 * n > (K - 256ll) * used : 48 * n > (K - 704ll) * used);
}

// ------------------------------------------------------------------------------------------------ gemm
// bf16, tiles of up to 256 rows x 256 weight rows (up: 128 gate rows and the 128 up rows beside them) x 64 per stage;
// weights are the A operand, so a lane holds one activation row and runs of four outputs.
// Bound by the LDS: 8 waves of 64 x 64 (the form before, 128 rows x 256) read a fragment per product, 128 bytes a cycle
// beside the stores; 4 waves of 128 x 128, one a SIMD, read half a fragment per product. A wave alone on its SIMD has to
// hide everything itself: fragments one sub-step ahead, loads two stages ahead, loads and LDS stores spread over the
// products (pinned: hipcc requests everything at a stage's end, 1182 us instead of 904 below), the barrier before the
// last sub-step. Tiles of fewer rows run 4 waves of 64 weight rows x all rows instead, in steps of 32.
// Narrow blocks (128 weight rows, tiles to 192 rows, two workgroups a CU) fill the chip with a quarter of the work.
// Both products of 4096 tokens, 16 experts of 3 x 4096 x 4096, top 2: 1143 -> 904 us (913 TFLOP/s without padding);
// 16 experts of 3 x 4096 x 2048, top 3: 764 -> 541; 1000 tokens, 32 experts of 3 x 2048 x 1024, top 4: 148 -> 116.
// Wide blocks where K % 64 == 0 go another way: expert_turns_tile.

// `bytes`: loads past them return zeros
__device__ __forceinline__ __amdgpu_buffer_rsrc_t uniform_rsrc(const void* p, unsigned bytes = ~0u) {
  const unsigned long long a = (unsigned long long)p;
  const unsigned long long u = ((unsigned long long)__builtin_amdgcn_readfirstlane((unsigned)(a >> 32)) << 32) |
                               (unsigned)__builtin_amdgcn_readfirstlane((unsigned)a);
  return __builtin_amdgcn_make_buffer_rsrc((void*)u, (short)0, (int)bytes, 0x00020000);
}

// The results of a wave's AI runs of 32 weight rows and BJ of 32 rows
template <bool UP, int WN, int AI, int WM, int BJ>
__device__ __forceinline__ void expert_store(const ExpertArgs& p, const f32x16 (&acc)[AI][BJ], int lo, int nr, int n0) {
  const int lane = threadIdx.x & 63, l32 = lane & 31, hh = lane >> 5, N = p.N;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wn = wv % WN, wm = wv / WN;
#pragma unroll
  for (int j = 0; j < BJ; ++j) {
    const int r = wm * BJ * 32 + j * 32 + l32;
    if (r >= nr) continue;
    const float s = p.scale ? p.wts[p.perm[lo + r]] : 1.f;
    bf16_t* y = reinterpret_cast<bf16_t*>(p.y) + (long long)(lo + r) * N;
#pragma unroll
    for (int i = 0; i < (UP ? AI / 2 : AI); ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int n = n0 + (wn * (UP ? AI / 2 : AI) + i) * 32 + 8 * q + 4 * hh;
        if (n >= N) continue;  // (N % 4 == 0)
        float o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if constexpr (UP) {
            const float gt = acc[i][j][4 * q + e] * s, up = acc[AI / 2 + i][j][4 * q + e] * s;
            o[e] = gt * __builtin_amdgcn_rcpf(1.f + __expf(-gt)) * up;
          } else {
            o[e] = acc[i][j][4 * q + e] * s;
          }
        }
        *reinterpret_cast<uint2*>(y + n) = make_uint2(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]));
      }
  }
}

// WN x WM waves, each with AI runs of 32 weight rows and BJ of 32 rows. FAR: addresses of 64 bits, for activations or an expert's
// weights that 32-bit byte offsets do not span
template <bool UP, int WN, int AI, int WM, int BJ, bool FAR = false, bool ONCE = false>
__device__ __forceinline__ void expert_gemm_tile(const ExpertArgs& p, bf16_t* gl, int ex, int lo, int nr, int n0) {
  constexpr int WP = WN * AI, RP = WM * BJ, NP = WP + RP;  // staging passes of 32 rows: weights, activations
  constexpr int STG = NP * 32 * GBK;                       // one stage (elements)
  static_assert(WN * WM == 4 && AI % 2 == 0, "four waves, gate runs beside up runs");
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), wn = wv % WN, wm = wv / WN;
  const int K = p.K, N = p.N;
  // staging: thread tid owns the 16-byte piece tid % 8 of rows tid / 8 + 32 i
  const int ch = tid & 7, sr = tid >> 3;
  const bf16_t* wb = reinterpret_cast<const bf16_t*>(p.w) + (long long)ex * (UP ? 2 * N : N) * K;
  const bf16_t* xb = reinterpret_cast<const bf16_t*>(p.x) + (UP ? 0ll : (long long)lo * K);
  constexpr unsigned OUT = 1u << 31;  // past the activations: a stage past K multiplies zeros
  const __amdgpu_buffer_rsrc_t rw = uniform_rsrc(wb), rx = uniform_rsrc(xb, OUT);
  const unsigned rb = FAR ? 1u : (unsigned)K * 2;  // FAR: wo and xo are row numbers
  unsigned wo[WP], xo[RP];
#pragma unroll
  for (int i = 0; i < WP; ++i) {
    const int r = sr + 32 * i;
    // (up: a wave's rows are AI / 2 runs of 32 gate rows, then the same up rows)
    const int run = r / 32, wrun = run % AI, base = run / AI * (AI / 2) * 32;
    const int n = UP ? (wrun < AI / 2 ? 0 : N) + min(n0 + base + wrun % (AI / 2) * 32 + (r & 31), N - 1) : min(n0 + r, N - 1);
    wo[i] = (unsigned)n * rb;
  }
#pragma unroll
  for (int i = 0; i < RP; ++i) {
    const int xr = min(sr + 32 * i, nr - 1);
    xo[i] = (unsigned)(UP ? p.perm[lo + xr] / p.top : xr) * rb;
  }
  u32x4 ra[2][NP];
  const int so = sr * GBK + ((ch ^ ((sr >> 1) & 7)) << 3);  // 16 rows x one piece cover all 64 banks
  auto load = [&](int t, int i, u32x4 (&r)[NP]) {
    const int k = t * GBK + ch * 8;
    if constexpr (FAR) {
      const bf16_t* row = i < WP ? wb + (long long)wo[i < WP ? i : 0] * K : xb + (long long)xo[i < WP ? 0 : i - WP] * K;
      const unsigned keep = i < WP || k < K ? ~0u : 0u;
      r[i] = *reinterpret_cast<const u32x4*>(row + min(k, K - 8)) & u32x4{keep, keep, keep, keep};
      return;
    }
    const unsigned kw = min(k, K - 8) * 2, kx = k < K ? k * 2 : OUT;
    const auto v = i < WP ? __builtin_amdgcn_raw_buffer_load_b128(rw, wo[i < WP ? i : 0] + kw, 0, ONCE ? 2 : 0)
                          : __builtin_amdgcn_raw_buffer_load_b128(rx, xo[i < WP ? 0 : i - WP] + kx, 0, 0);
    r[i] = *reinterpret_cast<const u32x4*>(&v);
  };
  auto store = [&](int i, bf16_t* buf, const u32x4 (&r)[NP]) {
    *reinterpret_cast<u32x4*>(buf + so + 32 * i * GBK) = r[i];
  };
  f32x16 acc[AI][BJ];
#pragma unroll
  for (int i = 0; i < AI; ++i)
#pragma unroll
    for (int j = 0; j < BJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  const int sw = (l32 >> 1) & 7;
  const int ar = (wn * AI * 32 + l32) * GBK, br = (WP * 32 + wm * BJ * 32 + l32) * GBK;
  const int nk = ((K + GBK - 1) / GBK + 1) & ~1;  // (an odd count's extra stage multiplies zeros)
  bf16x8 a[2][AI], x[2][BJ];
  auto frag = [&](const bf16_t* st, int s) {
#pragma unroll
    for (int i = 0; i < AI; ++i)
      a[s & 1][i] = *reinterpret_cast<const bf16x8*>(st + ar + i * 32 * GBK + (((2 * s + hh) ^ sw) << 3));
#pragma unroll
    for (int j = 0; j < BJ; ++j)
      x[s & 1][j] = *reinterpret_cast<const bf16x8*>(st + br + j * 32 * GBK + (((2 * s + hh) ^ sw) << 3));
  };
  auto products = [&](int s) {
#pragma unroll
    for (int i = 0; i < AI; ++i)
#pragma unroll
      for (int j = 0; j < BJ; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[s & 1][i], x[s & 1][j], acc[i][j], 0, 0, 0);
  };
  constexpr int NM = AI * BJ, NF = AI + BJ;  // products of a sub-step, its fragments
  // stage t: LDS buffer t & 1 holds it, register set (t + 1) & 1 the next, the other set the one after; a piece that is
  // stored makes room for its successor two stages on. The barrier
  // stands before the last sub-step, whose fragments are in registers: its products cover the first reads after it.
  auto stage = [&](int t, auto par) {
    constexpr int b = decltype(par)::value;
#pragma unroll
    for (int s = 0; s < 3; ++s) {
      constexpr int PP = (NP + 2) / 3;
      frag(gl + b * STG, s + 1);
#pragma unroll
      for (int i = s * PP; i < (s + 1) * PP && i < NP; ++i) {
        store(i, gl + (b ^ 1) * STG, ra[b ^ 1]);
        load(t + 3, i, ra[b ^ 1]);
      }
      products(s);
#pragma unroll
      for (int i = 0; i < NF; ++i) {  // (hipcc by itself requests everything at a stage's end)
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
      }
#pragma unroll
      for (int i = s * PP; i < (s + 1) * PP && i < NP; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x20, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x8, NM, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
    frag(gl + (b ^ 1) * STG, 0);
    products(3);
    __builtin_amdgcn_sched_group_barrier(0x100, NF, 0);
    __builtin_amdgcn_sched_group_barrier(0x8, NM, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
#pragma unroll
  for (int i = 0; i < NP; ++i) load(0, i, ra[0]);
#pragma unroll
  for (int i = 0; i < NP; ++i) load(1, i, ra[1]);
#pragma unroll
  for (int i = 0; i < NP; ++i) store(i, gl, ra[0]);
#pragma unroll
  for (int i = 0; i < NP; ++i) load(2, i, ra[0]);
  __syncthreads();
  frag(gl, 0);
  for (int t = 0; t < nk; t += 2) {
    stage(t, std::integral_constant<int, 0>{});
    stage(t + 1, std::integral_constant<int, 1>{});
  }
  expert_store<UP, WN, AI, WM, BJ>(p, acc, lo, nr, n0);
}

// A block's tile and weight block. An XCD works a contiguous run of (expert, weight block, row tile), so the row tiles that share a
// weight block are on one XCD at one time. Late tiles (late_tile: alone, at most half full, after all others) fill the CUs that the
// last long blocks leave idle.
struct GemmPlace {
  int tile, bn;
};
__device__ __forceinline__ GemmPlace gemm_place(const ExpertArgs& p, int nt, int nb) {
  int id = xcd_remap(blockIdx.x, nt * nb);
  const int* t0 = p.tiles + id / nb * 5;
  int first = t0[3], of = t0[4], large = 0;  // (requested with the count's loads; right where there are none)
  for (int i = 0; i < nt; i += 64) {
    const int t = i + (threadIdx.x & 63);
    const int* tl = p.tiles + min(t, nt - 1) * 5;
    large += __popcll(__ballot(t < nt && !(tl[4] == 1 && 2 * tl[2] <= p.mt)));
  }
  large = __builtin_amdgcn_readfirstlane(large);
  if (large > 0 && large < nt) {
    const int l = large * nb;
    id = (int)blockIdx.x < l ? xcd_remap(blockIdx.x, l) : l + xcd_remap(blockIdx.x - l, nt * nb - l);
    t0 = p.tiles + id / nb * 5;
    first = t0[3], of = t0[4];
  }
  const int in = id - first * nb;
  return {first + in % of, in / of};
}

// The tiles stand by size, largest first (group_rows). Of each size an XCD takes a run of neighbours, which share weight blocks or rows
// in its cache, and as much as the others. (One run of all sizes: the XCD of the largest tiles ends last, 4096 tokens above 834 us instead
// of 774. Rounds of 256 blocks over all XCDs: at 1200 tokens, whose tiles share nothing, eight neighbouring experts' gate and up rows
// at a time 437 instead of 386.) Returns -1 past the XCD's last.
__device__ __forceinline__ int turns_place(const ExpertArgs& p, int nt, int nb) {
  int n[4] = {0, 0, 0, 0};  // tiles of 4 .. 1 runs of 64 rows
  const int lane = threadIdx.x & 63;
  auto count = [&](int rows) {
#pragma unroll
    for (int b = 0; b < 4; ++b) n[b] += __popcll(__ballot((rows + 63) / 64 == 4 - b));
  };
  int i = 0;
  // Many tiles: eight loads at one time, as the block has nothing else to do. (One by one, both products of 1.9 million tokens, top 4, 16 experts of 3 x
  // 512 x 512, 29695 tiles, 126.6 ms, 120.7 in the four waves' blocks that were here before; so 42. 262144 tokens, 4111 tiles 6.4 -> 4.7.)
  for (; i + 512 <= nt; i += 512) {
    int rows[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) rows[j] = p.tiles[(i + 64 * j + lane) * 5 + 2];
#pragma unroll
    for (int j = 0; j < 8; ++j) count(rows[j]);
  }
  for (; i < nt; i += 64) count(i + lane < nt ? p.tiles[(i + lane) * 5 + 2] : 0);
  const int x = blockIdx.x & 7;
  int y = blockIdx.x >> 3, first = 0;
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const int m = __builtin_amdgcn_readfirstlane(n[b]) * nb, lo = (int)((long long)m * x >> 3), c = (int)((long long)m * (x + 1) >> 3) - lo;
    if (y < c) return first + lo + y;
    y -= c;
    first += m;
  }
  return -1;
}

template <bool UP>
__global__ void __launch_bounds__(512, 1) expert_turns_kernel(ExpertArgs p) {
  extern __shared__ __attribute__((aligned(1024))) char sl[];
  constexpr int NB = GN / (UP ? 2 : 1);
  const int nt = *p.ntiles, nb = (p.N + NB - 1) / NB;
  const int id = turns_place(p, nt, nb);
  if (id < 0) return;
  const int* t0 = p.tiles + id / nb * 5;
  const int in = id - t0[3] * nb, tile = t0[3] + in % t0[4], bn = in / t0[4];
  const int* tl = p.tiles + tile * 5;
  const int nr = tl[2], n0 = bn * NB;
  once_or_again(read_once(tl[4], tl[2], p.mt), [&](auto once) {
    constexpr bool ONCE = decltype(once)::value;
    if (nr > 192) expert_turns_tile<UP, 4>(p, sl, tl[0], tl[1], nr, n0);
    else if (nr > 128) expert_turns_tile<UP, 3, ONCE>(p, sl, tl[0], tl[1], nr, n0);
    else if (nr > 64) expert_turns_tile<UP, 2, ONCE>(p, sl, tl[0], tl[1], nr, n0);
    else expert_turns_tile<UP, 1, ONCE>(p, sl, tl[0], tl[1], nr, n0);
  });
}

// NARROW: tiles of up to 192 rows x 128 weight rows (FAR: 128 rows)
template <bool UP, bool NARROW, bool FAR = false>
__global__ void __launch_bounds__(256, NARROW ? 2 : 1) expert_gemm_kernel(ExpertArgs p) {
  extern __shared__ __attribute__((aligned(16))) bf16_t gl[];  // [2][weight rows, then activation rows][GBK]
  constexpr int NB = (NARROW ? 128 : 256) / (UP ? 2 : 1);
  const int nt = *p.ntiles, nb = (p.N + NB - 1) / NB;
  if ((int)blockIdx.x >= nt * nb) return;
  const GemmPlace at = gemm_place(p, nt, nb);
  const int* tl = p.tiles + at.tile * 5;
  const int nr = tl[2], n0 = at.bn * NB;
  if constexpr (FAR) {
    expert_gemm_tile<UP, 2, 2, 2, 2, true>(p, gl, tl[0], tl[1], nr, n0);
  } else if constexpr (NARROW) {
    once_or_again(read_once(tl[4], nr, p.mt), [&](auto once) {
      constexpr bool ONCE = decltype(once)::value;
      if (nr > 128) expert_gemm_tile<UP, 2, 2, 2, 3, false, ONCE>(p, gl, tl[0], tl[1], nr, n0);
      else if (nr > 64) expert_gemm_tile<UP, 2, 2, 2, 2, false, ONCE>(p, gl, tl[0], tl[1], nr, n0);
      else expert_gemm_tile<UP, 2, 2, 2, 1, false, ONCE>(p, gl, tl[0], tl[1], nr, n0);
    });
  } else {
    if (nr > 192) expert_gemm_tile<UP, 2, 4, 2, 4>(p, gl, tl[0], tl[1], nr, n0);
    else if (nr > 160) expert_gemm_tile<UP, 4, 2, 1, 6>(p, gl, tl[0], tl[1], nr, n0);
    else if (nr > 128) expert_gemm_tile<UP, 4, 2, 1, 5>(p, gl, tl[0], tl[1], nr, n0);
    else if (nr > 96) expert_gemm_tile<UP, 4, 2, 1, 4>(p, gl, tl[0], tl[1], nr, n0);
    else if (nr > 64) expert_gemm_tile<UP, 4, 2, 1, 3>(p, gl, tl[0], tl[1], nr, n0);
    else expert_gemm_tile<UP, 4, 2, 1, 2>(p, gl, tl[0], tl[1], nr, n0);
  }
}

template <bool UP, bool NARROW, bool FAR = false>
int gemm_go(const ExpertArgs& a, int max_tiles, hipStream_t s) {
  constexpr int NB = (NARROW ? 128 : 256) / (UP ? 2 : 1), LDS = NARROW ? GEMM_LDS / 8 * 5 : WIDE_LDS;
  auto kern = expert_gemm_kernel<UP, NARROW, FAR>;
  if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, LDS) != hipSuccess) return 5;
  hipLaunchKernelGGL(kern, dim3((a.N + NB - 1) / NB * max_tiles), dim3(256), LDS, s, a);
  return hipGetLastError() == hipSuccess ? 0 : 4;
}

template <bool UP>
int turns_go(const ExpertArgs& a, int max_tiles, hipStream_t s) {
  constexpr int NB = GN / (UP ? 2 : 1);
  auto kern = expert_turns_kernel<UP>;
  if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, WIDE_LDS) != hipSuccess) return 5;
  hipLaunchKernelGGL(kern, dim3((a.N + NB - 1) / NB * max_tiles + 32), dim3(512), WIDE_LDS, s, a);  // (an XCD's run of a size is one longer or not)
  return hipGetLastError() == hipSuccess ? 0 : 4;
}

template <typename E, bool VEC>
int gemv_go(const ExpertArgs& a, int mt, int max_tiles, hipStream_t s) {
  const int n = a.ws && a.Ns > a.N ? a.Ns : a.N;
  const dim3 g((n + (a.up ? 4 : 8) - 1) / (a.up ? 4 : 8), max_tiles + (a.ws ? (a.tokens + mt - 1) / mt : 0));
#define GO(M)                                                                                                  \
  do {                                                                                                         \
    constexpr int lds = M * 2048 * (int)sizeof(E);                                                             \
    auto kern = expert_gemv_kernel<E, M, VEC>;                                                                 \
    if (lds > 48 * 1024 &&                                                                                     \
        hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess) \
      return 5;                                                                                                \
    hipLaunchKernelGGL(kern, g, dim3(256), lds, s, a);                                                         \
  } while (0)
  if (mt == 1) GO(1);
  else if (mt == 2) GO(2);
  else if (mt == 4) GO(4);
  else if (mt == 8) GO(8);
  else return 6;
#undef GO
  return hipGetLastError() == hipSuccess ? 0 : 4;
}

bool al16(const void* p) { return (uintptr_t)p % 16 == 0; }

template <int NW, bool GROUP>
int route_lds(const RouteArgs& a) {
  const int zs = (a.E + (a.wsg ? 1 : 0) + 63) / 64 * 64;
  return ((a.softmax ? 3 : 1) * 16 * zs + NW * 1024 + (GROUP ? a.T * a.top : 0)) * 4;
}
constexpr int MAX_LDS = 160 * 1024;

// softmax routers: equal groups, enough experts in the kept ones
bool route_ok(const RouteArgs& a) {
  return a.T >= 1 && a.d >= 1 && a.E >= 1 && a.E <= 1024 && a.top >= 1 && a.top <= a.E && a.h && a.wr && a.ids && a.wts && (!a.wsg || a.sg) &&
         (!a.softmax || (a.groups >= 1 && a.E % a.groups == 0 && a.keep >= 1 && a.keep <= a.groups && a.top <= a.E / a.groups * a.keep));
}

template <int NW, bool GROUP>
int route_go(const RouteArgs& a, const GroupArgs& g, hipStream_t s) {
  const int lds = route_lds<NW, GROUP>(a);
  auto kern = route_mfma_kernel<NW, GROUP>;
  if (lds > 48 * 1024 && hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
    return 5;
  hipLaunchKernelGGL(kern, dim3((a.T + 15) / 16), dim3(NW * 64), lds, s, a, g);
  return hipGetLastError() == hipSuccess ? 0 : 4;
}

template <int GROUP>
int split_go(const RouteArgs& a, const GroupArgs& g, void* ws, long long ws_floats, void* cnt, int cnt_n, hipStream_t s) {
  const int n = a.E + (a.wsg ? 1 : 0), blocks = (a.T + 15) / 16;
  if (n > 64 || a.T > 1024 || !cnt || cnt_n < blocks + (GROUP == 2) || !al16(ws) || ws_floats < blocks * 256ll * ((n + 15) / 16 * 16)) return 6;
  hipLaunchKernelGGL(route_split_kernel<GROUP>, dim3(blocks * 4), dim3(1024), 0, s, a, g, (float*)ws, (unsigned*)cnt);
  return hipGetLastError() == hipSuccess ? 0 : 4;
}

}  // namespace

// dtype: 0 fp32, 1 bf16. ws: the split kernel (bf16, d % 8 == 0, up to 64 outputs with the shared gate and 1024 tokens), with
// ceil(T / 16) * 256 * (outputs rounded up to 16) floats there and ceil(T / 16) zeroed counters at cnt (left zeroed)
KCA_API int kca_moe_route(int dtype, const void* h, const void* wr, const void* wsg, void* ids, void* wts, void* sg,
                          int T, int d, int E, int top, int softmax, const void* fix, int groups, int keep, void* ws,
                          long long ws_floats, void* cnt, int cnt_n, hipStream_t s) {
  const RouteArgs a{h, wr, wsg, (int*)ids, (float*)wts, (float*)sg, T, d, E, top, softmax, groups, keep, (const float*)fix};
  if (!route_ok(a)) return 1;
  if (dtype == 1 && d % 8 == 0 && al16(h) && al16(wr) && al16(wsg)) {
    if (ws) return split_go<0>(a, GroupArgs{}, ws, ws_floats, cnt, cnt_n, s);
    if (T <= 1024 && route_lds<16, false>(a) <= MAX_LDS) return route_go<16, false>(a, GroupArgs{}, s);
    if (route_lds<8, false>(a) <= MAX_LDS) return route_go<8, false>(a, GroupArgs{}, s);
  }
  const int lds = ((softmax ? 3 : 1) * E + 1) * 4;
  if (dtype == 1) hipLaunchKernelGGL(route_rows_kernel<bf16_t>, dim3(T), dim3(256), lds, s, a);
  else if (dtype == 0) hipLaunchKernelGGL(route_rows_kernel<float>, dim3(T), dim3(256), lds, s, a);
  else return 3;
  return hipGetLastError() == hipSuccess ? 0 : 4;
}

static bool group_ok(const GroupArgs& g, int max_tiles) {
  return g.n >= 1 && g.E >= 1 && g.E <= 1024 && g.mt >= 1 && g.ids && g.perm && g.inv && g.tiles && g.ntiles &&
         max_tiles >= (g.E < g.n ? g.E : g.n) + g.n / g.mt;
}

// tiles: [max_tiles][5] with max_tiles >= min(E, n) + n / mt
KCA_API int kca_moe_group(const void* ids, int n, int E, int mt, void* perm, void* inv, void* tiles, int max_tiles,
                          void* ntiles, hipStream_t s) {
  const GroupArgs g{(const int*)ids, n, E, mt, (int*)perm, (int*)inv, (int*)tiles, (int*)ntiles};
  if (!group_ok(g, max_tiles)) return 1;
  hipLaunchKernelGGL(group_kernel, dim3(1), dim3(1024), (4 * E + 3) * 4, s, g);
  return hipGetLastError() == hipSuccess ? 0 : 4;
}

// Both in one launch: bf16, at most 16 tokens, or with ws (kca_moe_route; one counter more) 1024 (10: shape outside it). E: router
// outputs, the first `real` with weights
KCA_API int kca_moe_route_group(const void* h, const void* wr, const void* wsg, void* ids, void* wts, void* sg, int T,
                                int d, int E, int real, int top, int softmax, const void* fix, int groups, int keep, int mt, void* perm,
                                void* inv, void* tiles, int max_tiles, void* ntiles, void* ws, long long ws_floats, void* cnt,
                                int cnt_n, hipStream_t s) {
  const RouteArgs a{h, wr, wsg, (int*)ids, (float*)wts, (float*)sg, T, d, E, top, softmax, groups, keep, (const float*)fix};
  if (!route_ok(a) || real < 1 || real > E) return 1;
  if (T > (ws ? 1024 : 16) || top > 64 || d % 8 || !al16(h) || !al16(wr) || !al16(wsg) || (!ws && route_lds<16, true>(a) > MAX_LDS)) return 10;
  const GroupArgs g{(const int*)ids, T * top, real, mt, (int*)perm, (int*)inv, (int*)tiles, (int*)ntiles};
  if (!group_ok(g, max_tiles)) return 1;
  if (ws) return T > 16 ? split_go<2>(a, g, ws, ws_floats, cnt, cnt_n, s) : split_go<1>(a, g, ws, ws_floats, cnt, cnt_n, s);
  return route_go<16, true>(a, g, s);
}

// One expert product of every tile. mt: the tiles' row limit (1, 2, 4, 8: gemv; 32: stream, bf16 with K % 64 == 0 and
// N % 16 == 0; 128, 192, 256: gemm, bf16 with K % 8 == 0 and N % 4 == 0). x_rows: rows of x. Where the rows that a tile gathers span
// 2 GiB or an expert's weights 4 GiB, gemm tiles have up to 128 rows. ws: a shared expert's product over all tokens beside
// them (gemv; nullable).
KCA_API int kca_moe_expert(int dtype, const void* x, const void* w, void* y, const void* perm, const void* wts,
                           const void* tiles, const void* ntiles, int max_tiles, int mt, int top, int N, int K, int up,
                           int scale, const void* xs, const void* ws, void* ys, int tokens, int Ns, int Ks, int x_rows,
                           hipStream_t s) {
  if (max_tiles < 1 || max_tiles > 32767 || N < 1 || K < 1 || top < 1 || !x || !w || !y || !perm || !wts || !tiles || !ntiles) return 1;
  if (ws && (!xs || !ys || tokens < 1 || tokens > 32767 || Ns < 1 || Ks < 1 || mt > 8)) return 1;
  const ExpertArgs a{x, w, y, (const int*)perm, (const float*)wts, (const int*)tiles, (const int*)ntiles, mt, top, N, K, up, scale,
                     xs, ws, ys, tokens, Ns, Ks};
  const bool far = (up ? 4ll : 2ll) * N * K >= 1ll << 32 || 2ll * (up ? x_rows : mt) * K >= 1ll << 31;  // (32-bit byte offsets)
  if (mt == GM || mt == 128 || mt == 192) {
    if (dtype != 1 || K % 8 || N % 4 || !al16(x) || !al16(w) || (uintptr_t)y % 8 || (far && mt != 128)) return 10;
    if (far) return up ? gemm_go<true, true, true>(a, max_tiles, s) : gemm_go<false, true, true>(a, max_tiles, s);
    if (mt == GM && K % GBK == 0) return up ? turns_go<true>(a, max_tiles, s) : turns_go<false>(a, max_tiles, s);
    if (mt == GM) return up ? gemm_go<true, false>(a, max_tiles, s) : gemm_go<false, false>(a, max_tiles, s);
    return up ? gemm_go<true, true>(a, max_tiles, s) : gemm_go<false, true>(a, max_tiles, s);
  }
  if (mt == SROWS) {
    if (dtype != 1 || K % SK || N % 16 || !al16(x) || !al16(w) || (uintptr_t)y % 8 || far) return 10;
    const bool block = stream_block(up, N, K, top, x_rows, max_tiles);
    auto kern = block ? (up ? expert_block_kernel<true> : expert_block_kernel<false>) : (up ? expert_stream_kernel<true> : expert_stream_kernel<false>);
    if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, STREAM_LDS) != hipSuccess) return 5;
    const int nb = (block ? BWN : SWN) / (up ? 2 : 1);
    const long long blocks = (N + nb - 1ll) / nb * max_tiles;
    if (blocks >= 1ll << 31) return 10;
    hipLaunchKernelGGL(kern, block_rows(blocks), dim3(256), STREAM_LDS, s, a);
    return hipGetLastError() == hipSuccess ? 0 : 4;
  }
  const int v = dtype == 1 ? 8 : 4;
  const bool vec = K % v == 0 && al16(x) && al16(w) && (!ws || (Ks % v == 0 && al16(xs) && al16(ws)));
  if (dtype == 0) return vec ? gemv_go<float, true>(a, mt, max_tiles, s) : gemv_go<float, false>(a, mt, max_tiles, s);
  if (dtype == 1) return vec ? gemv_go<bf16_t, true>(a, mt, max_tiles, s) : gemv_go<bf16_t, false>(a, mt, max_tiles, s);
  return 3;
}
