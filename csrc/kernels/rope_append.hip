// Prompt rows into the serving cache: rotates Q and K of a fused projection in place and writes K (rotated) and V into
// their pages (or contiguous slots), one launch a layer.
//
// Bound by memory: K and V are read and written once, the rotated part of Q read and written. 32 lanes own one
// (token, head) row, 16 bytes each, so every load and store is a whole line and a row's rotation partners sit in one
// wave (a row's loads are all issued before its first store). It replaces a rotation launch, two gathers of the
// unpadded rows and two index scatters: 6 prompts of 700 to 1100 tokens, 16 heads of 256: 225 -> 62 us a layer; a
// workgroup over one token's rows, 8 or 24 in flight, measured 61 and 68. With a row, its place and its factors requested together, not
// each behind a test of the one before, 57 -> 49 us (210 MB at 4.3 TB/s), 1500 tokens x 64 heads of 96 67 -> 59.
#include "common.h"

namespace {

struct AppendArgs {
  bf16_t *q, *k;        // 16-bit elements of either type
  const bf16_t* v;
  long long q_st, q_sh, k_st, k_sh, v_st, v_sh;
  int T, H, Hkv, D, rot, interleaved;
  const float *cs, *sn;           // [positions][rot / 2]
  const int *pos, *page, *off;    // [T]: position, page (slot) and row in it; page < 0: the row is padding
  bf16_t *kc, *vc;                // [pages][Hkv][per][D]
  int per;
};

template <bool F16> __device__ __forceinline__ float to_f(bf16_t x) {
  if constexpr (F16) return (float)*reinterpret_cast<const _Float16*>(&x);
  else return bf2f(x);
}
template <bool F16> __device__ __forceinline__ bf16_t from_f(float x) {
  if constexpr (F16) {
    const _Float16 h = (_Float16)x;
    return *reinterpret_cast<const bf16_t*>(&h);
  } else {
    return f2bf(x);
  }
}

struct __attribute__((aligned(16))) Chunk { bf16_t e[8]; };

// A workgroup is one head row of 8 tokens: 4 KiB of a page that lie together.
template <bool F16>
__global__ void __launch_bounds__(256) rope_append_kernel(AppendArgs a) {
  const int lane = threadIdx.x & 31, nq = a.rot > 0 ? a.H : 0, heads = nq + 2 * a.Hkv;
  const int j = blockIdx.x % heads, t = blockIdx.x / heads * 8 + (threadIdx.x >> 5), d = lane * 8;
  if (t >= a.T || d >= a.D) return;
  const bool is_q = j < nq, is_v = j >= nq + a.Hkv;
  const int h = is_q ? j : is_v ? j - nq - a.Hkv : j - nq;
  if (is_q && d >= a.rot) return;
  bf16_t* src = is_q ? a.q + t * a.q_st + h * a.q_sh : is_v ? const_cast<bf16_t*>(a.v) + t * a.v_st + h * a.v_sh
                                                            : a.k + t * a.k_st + h * a.k_sh;
  // (the row and where it goes are requested together: a test of the page first costs a second round trip)
  Chunk x = *reinterpret_cast<const Chunk*>(src + d);
  const int page = a.page[t], off = a.off[t];
  if (!is_v && d < a.rot) {
    const int half = a.rot >> 1, pos = a.pos[t];
    const float *cs = a.cs + (long long)pos * half, *sn = a.sn + (long long)pos * half;
    // (factors past the rotated part are the last ones, unused: loads behind conditions would follow each other)
    if (a.interleaved) {  // pairs (2i, 2i + 1)
      float c[4], n[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) c[i] = cs[min(d / 2 + i, half - 1)], n[i] = sn[min(d / 2 + i, half - 1)];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float u = to_f<F16>(x.e[2 * i]), w = to_f<F16>(x.e[2 * i + 1]);
        // (which product is rounded first is written out: the compiler's choice hangs on the code around it)
        const bf16_t p = from_f<F16>(fmaf(u, c[i], -(w * n[i]))), r = from_f<F16>(fmaf(u, n[i], w * c[i]));
        if (d + 2 * i < a.rot) x.e[2 * i] = p, x.e[2 * i + 1] = r;
      }
    } else {  // pairs (i, i + rot / 2): the partners are read before any lane of the row stores
      Chunk y;
      float c[8], n[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int e = min(d + i, a.rot - 1), p = e < half ? e : e - half;
        c[i] = cs[p], n[i] = e < half ? -sn[p] : sn[p];
      }
      if (half % 8 == 0) {
        y = *reinterpret_cast<const Chunk*>(src + (d < half ? d + half : d - half));
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int e = min(d + i, a.rot - 1);
          y.e[i] = src[e < half ? e + half : e - half];
        }
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const bf16_t r = from_f<F16>(fmaf(to_f<F16>(x.e[i]), c[i], to_f<F16>(y.e[i]) * n[i]));
        if (d + i < a.rot) x.e[i] = r;
      }
    }
    *reinterpret_cast<Chunk*>(src + d) = x;
  }
  if (is_q || page < 0) return;
  bf16_t* dst = (is_v ? a.vc : a.kc) + (((long long)page * a.Hkv + h) * a.per + off) * a.D + d;
  *reinterpret_cast<Chunk*>(dst) = x;
}

bool rows16(const void* p, long long st, long long sh) { return (uintptr_t)p % 16 == 0 && (st | sh) % 8 == 0; }

}  // namespace

// dtype: 1 bf16, 2 fp16. Returns 1 for rows that 16-byte chunks do not fit (the caller takes its general way).
KCA_API int kca_rope_append(int dtype, void* q, void* k, const void* v, long long q_st, long long q_sh, long long k_st,
                            long long k_sh, long long v_st, long long v_sh, int T, int H, int Hkv, int D, int rot,
                            int interleaved, const float* cs, const float* sn, const int* pos, const int* page,
                            const int* off, void* kc, void* vc, int per, hipStream_t stream) {
  if ((dtype != 1 && dtype != 2) || T < 1 || D % 8 || D < 8 || D > 256 || rot % 2 || rot < 0 || rot > D || per < 1) return 1;
  if (!rows16(q, q_st, q_sh) || !rows16(k, k_st, k_sh) || !rows16(v, v_st, v_sh) || !rows16(kc, 0, 0) || !rows16(vc, 0, 0))
    return 1;
  const AppendArgs a{(bf16_t*)q, (bf16_t*)k, (const bf16_t*)v, q_st, q_sh, k_st, k_sh, v_st, v_sh, T, H, Hkv, D, rot,
                     interleaved, cs, sn, pos, page, off, (bf16_t*)kc, (bf16_t*)vc, per};
  const dim3 grid((unsigned)((T + 7) / 8 * ((rot > 0 ? H : 0) + 2 * Hkv)));
  if (dtype == 2) hipLaunchKernelGGL(rope_append_kernel<true>, grid, dim3(256), 0, stream, a);
  else hipLaunchKernelGGL(rope_append_kernel<false>, grid, dim3(256), 0, stream, a);
  return hipGetLastError() == hipSuccess ? 0 : 4;
}
