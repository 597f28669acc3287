// Fused per-head RMSNorm + rotary embedding of q and k, the producer step just
// before attention in Qwen3Attention.forward (qwen3.py:91-105):
//   q = RMSNorm(q per head) * q_norm.weight      layernorm.py:17-27 (rms_forward)
//   k = RMSNorm(k per head) * k_norm.weight
//   q, k = rotary_emb(positions, q, k)           rotary_embedding.py:6-17, 37-55
// With no norm weights it is the rotary embedding alone (Qwen2, qwen2.py:91-92).
//
// A wave takes 64/LPR head rows of one token (LPR = D/16 lanes per row), or kChunks times as
// many.  Lane j of a row holds 8 consecutive elements of each half of the head dimension,
// [8 j, 8 j + 8) and [D/2 + 8 j, ...), so the rotation pairs (i, i + D/2) are
// lane-local and only the sum of squares crosses lanes (xor shuffles over LPR
// lanes).
//
// What bounds a large launch: HBM (each row is read once and written once).  So a lane moves 16
// bytes per access and issues all its rows' loads before any of them is used (4 KiB in
// flight per wave at D = 128), the token's cos/sin row is loaded once for all of a
// wave's heads (per head it is twice the bytes of the row itself, through L1), and no
// index needs a division.  Stores are non-temporal.  8813 tokens, heads 32/8, D = 128 (185 MB):
// 46.4 us with 8-byte accesses, one row per lane group and cos/sin per head; 40.5 us in
// this form with 3 chunks per wave, 39.9 with 2, 42.2 with 1, 46.4 with 5; with the
// non-temporal stores 35.2 us = 5.26 TB/s (a 2 GiB device copy: 4.9 TB/s).  With the
// attention that reads q and k right after: a prefill of those tokens 269.5 -> 270.9 us,
// a decode of 128 rows 34.3 -> 34.0 us (producer and attention together, plain against
// non-temporal).
//
// A small launch (up to kSmallRows rows: every decode step) is bound by one wave's latency:
// one chunk per wave, half the code, and the norm weights loaded with the rows instead of
// after the reduction that needs them.  Captured, heads 16/8 with norm, 2 chunks -> 1: 1 token
// 3.0 -> 2.5 us, 33 3.4 -> 2.75, 256 3.5 -> 2.9; heads 32/8, 256 tokens 3.7 -> 3.3 (10240
// rows), 512 4.0 -> 4.2 (20480), hence the line.
//
// Arithmetic follows the reference's eager op sequence, rounding where it
// rounds: fp32 x, mean of squares, x * rsqrt(mean + eps) rounded to bf16, times
// the bf16 weight rounded to bf16; then fp32 x1*cos - x2*sin and x2*cos + x1*sin
// with every product and sum rounded separately (no FMA contraction), rounded
// to bf16.  The sum of squares runs in this kernel's order (a lane's squares,
// then a butterfly over the row's lanes), which can move the mean by an fp32 ulp against
// torch's reduction and so, rarely, an output by one bf16 ulp.
#include "nva_common.h"
#include "nva_kernels.h"

namespace nva {

namespace {

constexpr int kChunks = 2;         // head chunks of a token that one wave takes
constexpr int64_t kSmallRows = 16384;  // head rows up to which a launch is bound by latency
constexpr int kTokensPerGroup = 4;  // waves per workgroup, one token each
constexpr int64_t kMaxGroups = int64_t{1} << 22;  // tokens beyond 4 per workgroup: further rounds of the grid

// 8 bf16 of a row: one 16-byte access, or four of 4 bytes where a pointer or a row
// stride does not allow it.
template <bool WIDE>
__device__ __forceinline__ u32x4 load8(const uint16_t* p) {
  if constexpr (WIDE) return ld16(p);
  const uint32_t* w = reinterpret_cast<const uint32_t*>(p);
  return u32x4{w[0], w[1], w[2], w[3]};
}
template <bool WIDE, bool NT>
__device__ __forceinline__ void store8(uint16_t* p, u32x4 v) {
  if constexpr (WIDE && NT) {
    __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(p));
  } else if constexpr (WIDE) {
    st16(p, v);
  } else {
    uint32_t* w = reinterpret_cast<uint32_t*>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = v[i];
  }
}
template <bool WIDE>
__device__ __forceinline__ void load8f(const float* p, float (&f)[8]) {
  if constexpr (WIDE) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(p), b = *reinterpret_cast<const f32x4*>(p + 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f[i] = a[i];
      f[4 + i] = b[i];
    }
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) f[i] = p[i];
  }
}

__device__ __forceinline__ void unpack8(u32x4 w, float (&f)[8]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = bf16_bits_to_f32(w[i] & 0xffffu);
    f[2 * i + 1] = __builtin_bit_cast(float, w[i] & 0xffff0000u);
  }
}

// Round 8 values to bf16.
__device__ __forceinline__ void round8(float (&f)[8]) {
  u32x4 w;
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] = pack_bf16x2(f[2 * i], f[2 * i + 1]);
  unpack8(w, f);
}

}  // namespace

template <int D, bool WIDE, int CHUNKS, bool NT>
__global__ __launch_bounds__(64 * kTokensPerGroup) void qk_norm_rope_kernel(QKNormRopeParams p) {
  // every product and sum rounds on its own, as the reference's separate ops do:
  // no FMA contraction anywhere in this function
#pragma clang fp contract(off)
  constexpr int LPR = D / 16;      // lanes per row
  constexpr int RPW = 64 / LPR;    // rows (heads) per wave and chunk
  const int lane = threadIdx.x & 63;
  const int j = lane & (LPR - 1);
  const int heads = p.num_heads + p.num_kv_heads;
  const int h0 = static_cast<int>(blockIdx.y) * CHUNKS * RPW;
  const int64_t step = static_cast<int64_t>(gridDim.x) * kTokensPerGroup;
  for (int64_t t = static_cast<int64_t>(blockIdx.x) * kTokensPerGroup +
                   __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
       t < p.num_tokens; t += step) {
    int64_t pos = p.positions[t];
    const uint16_t* src[CHUNKS];
    uint16_t* dst[CHUNKS];
    u32x4 lo[CHUNKS], hi[CHUNKS];
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      const int hh = h0 + c * RPW + lane / LPR;
      const bool is_q = hh < p.num_heads;
      src[c] = is_q ? p.q + t * p.q_row_stride + hh * D : p.k + t * p.k_row_stride + (hh - p.num_heads) * D;
      dst[c] = is_q ? p.q_out + t * p.q_out_row_stride + hh * D
                    : p.k_out + t * p.k_out_row_stride + (hh - p.num_heads) * D;
      lo[c] = hi[c] = u32x4{0u, 0u, 0u, 0u};
      if (hh < heads) {
        lo[c] = load8<WIDE>(src[c] + 8 * j);
        hi[c] = load8<WIDE>(src[c] + D / 2 + 8 * j);
      }
    }
    u32x4 wlo = {0u, 0u, 0u, 0u}, whi = {0u, 0u, 0u, 0u};
    if constexpr (CHUNKS == 1) {
      if (p.q_weight) {
        const uint16_t* wt = h0 + lane / LPR < p.num_heads ? p.q_weight : p.k_weight;
        wlo = load8<WIDE>(wt + 8 * j);
        whi = load8<WIDE>(wt + D / 2 + 8 * j);
      }
    }
    // cache row = [cos(D/2) | sin(D/2)] of the clamped position
    pos = pos < 0 ? 0 : (pos >= p.max_position ? p.max_position - 1 : pos);
    float cs[8], sn[8];
    load8f<WIDE>(p.cos_sin + pos * D + 8 * j, cs);
    load8f<WIDE>(p.cos_sin + pos * D + D / 2 + 8 * j, sn);
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      if (h0 + c * RPW >= heads) break;  // uniform: the whole chunk lies past the last head
      const int hh = h0 + c * RPW + lane / LPR;
      float x1[8], x2[8];
      unpack8(lo[c], x1);
      unpack8(hi[c], x2);
      if (p.q_weight) {  // RMSNorm over the head dimension (uniform branch)
        float ss = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) ss = (ss + x1[e] * x1[e]) + x2[e] * x2[e];
#pragma unroll
        for (int m = LPR / 2; m >= 1; m >>= 1) ss += __shfl_xor(ss, m, LPR);
        const float r = rsqrtf(ss / static_cast<float>(D) + p.eps);
        if constexpr (CHUNKS > 1) {
          const uint16_t* wt = hh < p.num_heads ? p.q_weight : p.k_weight;
          wlo = load8<WIDE>(wt + 8 * j);
          whi = load8<WIDE>(wt + D / 2 + 8 * j);
        }
        float w1[8], w2[8];
        unpack8(wlo, w1);
        unpack8(whi, w2);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          x1[e] *= r;
          x2[e] *= r;
        }
        round8(x1);
        round8(x2);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          x1[e] *= w1[e];
          x2[e] *= w2[e];
        }
        round8(x1);
        round8(x2);
      }
      u32x4 o1, o2;
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        float y1[2], y2[2];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const int e = 2 * w + b;
          y1[b] = x1[e] * cs[e] - x2[e] * sn[e];
          y2[b] = x2[e] * cs[e] + x1[e] * sn[e];
        }
        o1[w] = pack_bf16x2(y1[0], y1[1]);
        o2[w] = pack_bf16x2(y2[0], y2[1]);
      }
      if (hh < heads) {
        store8<WIDE, NT>(dst[c] + 8 * j, o1);
        store8<WIDE, NT>(dst[c] + D / 2 + 8 * j, o2);
      }
    }
  }
}

// The wide accesses need 16-byte aligned rows, weights and table (rows of every engine
// tensor are); other inputs take 4-byte accesses of the same kernel.
static bool rows_aligned16(const QKNormRopeParams& p) {
  auto a = [](const void* x) { return reinterpret_cast<uintptr_t>(x) % 16 == 0; };
  return a(p.q) && a(p.k) && a(p.q_out) && a(p.k_out) && a(p.q_weight) && a(p.k_weight) && a(p.cos_sin) &&
         (p.q_row_stride | p.k_row_stride | p.q_out_row_stride | p.k_out_row_stride) % 8 == 0;
}

hipError_t launch_qk_norm_rope(const QKNormRopeParams& p, hipStream_t stream) {
  const int heads = p.num_heads + p.num_kv_heads;
  if (p.num_tokens <= 0 || heads <= 0) return hipSuccess;
  const int chunk = 64 / (p.head_dim / 16);  // heads
  const bool small = p.num_tokens * heads <= kSmallRows;
  const int per_wave = small ? chunk : kChunks * chunk;
  const int64_t groups = (p.num_tokens + kTokensPerGroup - 1) / kTokensPerGroup;
  const dim3 grid(static_cast<unsigned>(groups < kMaxGroups ? groups : kMaxGroups),
                  static_cast<unsigned>((heads + per_wave - 1) / per_wave));
  const dim3 block(64 * kTokensPerGroup);
  const bool wide = rows_aligned16(p);
#define NVA_ROPE(DD, WD, CH, NT) hipLaunchKernelGGL((qk_norm_rope_kernel<DD, WD, CH, NT>), grid, block, 0, stream, p)
#define NVA_ROPE_D(DD)                                     \
  do {                                                     \
    if (!wide && small) NVA_ROPE(DD, false, 1, false);       \
    else if (!wide) NVA_ROPE(DD, false, kChunks, false);   \
    else if (small) NVA_ROPE(DD, true, 1, false);          \
    else NVA_ROPE(DD, true, kChunks, true);                \
  } while (0)
  if (p.head_dim == 128) NVA_ROPE_D(128);
  else NVA_ROPE_D(64);
#undef NVA_ROPE_D
#undef NVA_ROPE
  return hipGetLastError();
}

}  // namespace nva
