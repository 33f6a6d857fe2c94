// Arguments and device helpers shared by the fused forward kernels
// (htree_fwd.hip, htree_fwd_stream.hip, htree_fwd_wide.h).
#pragma once

#include "htree_common.h"

namespace htree {

// max of a level that accumulated nothing (src/naive.py:9, src/parallel.py:75)
constexpr float kNegInfSentinel = -1.0e10f;

struct FwdArgs {
  LevelPtrs lv[HTREE_MAX_LEVELS];
  const void* q;
  void* out;
  float* gmax;
  float* gsum;
  int32_t* parents;
  uint16_t* scores;  // nullable: fp16 S - m_ref per (level, group, tile) for the backward
  float* smref;      // m_ref per (level, group, head)
  float* tmax;       // trace (TRACE kernels only): each level's own state,
  float* tsum;       //   [L, B, T, H] max / sum and [L, B, T, H, D] output
  float* tout;
  const float* cosb;
  const float* sinb;
  int32_t B, T, H, Hkv, G, CR, crlg, TK, L, max_tiles;
  float scale;
  int32_t per_xcd;
  int32_t kv_share;  // 2 or 4: KV heads kv_share*i .. kv_share*i + kv_share - 1 share one selection
  int32_t gpad;      // padding heads at the end of the group of KV heads h, h % kv_share == kv_share - 1
};

// query heads of KV head h that take part in the selection (the group's
// heads but the padding of the last KV head of a shared selection)
__device__ __forceinline__ int sel_heads(const FwdArgs& a, int h) {
  return a.G - ((h & (a.kv_share - 1)) == a.kv_share - 1 ? a.gpad : 0);  // kv_share 1, 2, 4
}

// The query (dslot's order) turned in place by the angle of cosr / sinr.  D >= 64: each pair
// (lo, hi) in one lane becomes (lo c - hi s, hi c + lo s), the products
// hi s and lo s rounded first, then one fma each: the arithmetic the
// compiler emits for rope_frag, but written in place, since the C form gets
// new registers for the turned query and pays a register move per value at
// every turn of the scoring loop (32 at D = 128).
template <int D>
__device__ __forceinline__ void rot_by(float (&x)[D / 32][8], const float* __restrict__ cosr,
                                       const float* __restrict__ sinr, int kg) {
  if constexpr (D == 32) {
    rope_frag32_lanes(x, cosr, sinr, kg, x);
  } else {
    constexpr int SPH = D / 64;
#pragma unroll
    for (int m = 0; m < SPH; ++m) {
      const int i0 = dslot<D>(kg, m);
      float c[8], s[8];
      Io<float>::ld8(cosr + i0, c);
      Io<float>::ld8(sinr + i0, s);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float lo = x[m][e], hi = x[m + SPH][e], ta, tb;
        asm("v_mul_f32 %2, %1, %4\n\t"
            "v_mul_f32 %3, %0, %4\n\t"
            "v_fma_f32 %0, %0, %5, -%2\n\t"
            "v_fma_f32 %1, %1, %5, %3"
            : "+v"(lo), "+v"(hi), "=&v"(ta), "=&v"(tb)
            : "v"(s[e]), "v"(c[e]));
        x[m][e] = lo;
        x[m + SPH][e] = hi;
      }
    }
  }
}

template <int D>
__device__ __forceinline__ void to_bf(const float (&x)[D / 32][8], bf16x8 (&h)[D / 32]) {
#pragma unroll
  for (int m = 0; m < D / 32; ++m) h[m] = pack8(x[m]);
}

template <int D>
__device__ __forceinline__ void to_bf_split(const float (&x)[D / 32][8], bf16x8 (&h)[D / 32],
                                            bf16x8 (&lo)[D / 32]) {
#pragma unroll
  for (int m = 0; m < D / 32; ++m) split8(x[m], h[m], lo[m]);
}

// ---------------------------------------------------------------- level trace
// The TRACE kernels start every level from an empty softmax state, so after
// the level (m, l, O) is that level's own state (LayerTrace of
// src/naive.py:13-19, filled at :225-227): max and output relative to the
// max over the level's accumulated candidates, -1e10 / 0 / 0 where the level
// accumulated nothing.  O[n][r] is output dim odim(n, 4kg + r) of head u16.
// Output dim of row i of O tile n: tiles 2j and 2j + 1 hold the even and the
// odd dims of 32j .. 32j + 31, so that the V^T fragments of a tile pair are one
// 16-byte load.
__device__ __forceinline__ int odim(int n, int i) { return 32 * (n >> 1) + 2 * i + (n & 1); }

// The head's output row from its O tiles (odim): a lane's values of a
// tile pair are the 8 consecutive dims 32j + 8kg .. + 7, stored as 16 bytes
// (against 2-byte stores: T 131072, 64/8 heads -1.3%; T 32768 within 0.3%).
template <int D, typename TIn, typename F>
__device__ __forceinline__ void store_out(TIn* op, int kg, const f32x4 (&O)[D / 16], F norm) {
#pragma unroll
  for (int j = 0; j < D / 32; ++j) {
    float x[8];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      x[2 * r] = norm(O[2 * j][r]);
      x[2 * r + 1] = norm(O[2 * j + 1][r]);
    }
    Io<TIn>::st8(op + 32 * j + 8 * kg, x);
  }
}

template <int D>
__device__ __forceinline__ void trace_store(const FwdArgs& a, int l, int64_t hq, bool gv, int kg,
                                            float m, float lpart, const f32x4 (&O)[D / 16]) {
  const float lt = add_xor32(add_xor16(lpart));
  if (!gv) return;
  const int64_t lh = (int64_t)l * a.B * a.T * a.H + hq;
  float* op = a.tout + lh * D;
#pragma unroll
  for (int n = 0; n < D / 16; ++n)
#pragma unroll
    for (int r = 0; r < 4; ++r) op[odim(n, 4 * kg + r)] = O[n][r];
  if (kg == 0) {
    a.tmax[lh] = m == -INFINITY ? kNegInfSentinel : m;
    a.tsum[lh] = lt;
  }
}

// Merges the levels' states top -> bottom with the guards of
// src/naive.py:215-223 (a state counts only where its sum > 1e-10); returns
// the merged sum, the merged max in m and output in O.  Reads back what this
// lane's trace_store calls wrote.
template <int D>
__device__ __forceinline__ float trace_merge(const FwdArgs& a, int64_t hq, bool gv, int kg,
                                             float& m, f32x4 (&O)[D / 16]) {
  float gm = kNegInfSentinel, gs = 0.f;
#pragma unroll
  for (int n = 0; n < D / 16; ++n) O[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (gv) {
    for (int l = a.L - 1; l >= 0; --l) {
      const int64_t lh = (int64_t)l * a.B * a.T * a.H + hq;
      const float lm = a.tmax[lh], ls = a.tsum[lh];
      if (!(ls > 1e-10f)) continue;
      const float* op = a.tout + lh * D;
      if (gs > 1e-10f) {
        const float nm = fmaxf(gm, lm);
        const float sg = expf(gm - nm), sc = expf(lm - nm);
        gs = gs * sg + ls * sc;
#pragma unroll
        for (int n = 0; n < D / 16; ++n)
#pragma unroll
          for (int r = 0; r < 4; ++r) O[n][r] = O[n][r] * sg + op[odim(n, 4 * kg + r)] * sc;
        gm = nm;
      } else {
        gs = ls;
#pragma unroll
        for (int n = 0; n < D / 16; ++n)
#pragma unroll
          for (int r = 0; r < 4; ++r) O[n][r] = op[odim(n, 4 * kg + r)];
        gm = lm;
      }
    }
  }
  m = gm;
  return gs;
}

// The launches of the streaming forward (levels of 17..64 candidate tiles,
// or groups with padding heads) and of the wide forward (top_k > 64, more
// than 64 tiles, or KV-head quads); sel: the selection-only instances.
void launch_fwd_stream(int D, int dtype, const FwdArgs& a, dim3 grid, hipStream_t st, bool sel);
template <int D>
void launch_fwd_wide_d(int dtype, const FwdArgs& a, dim3 grid, hipStream_t st, bool sel);

// fn(PREC, (TIn*)) for the input types, fn(D, PREC, (TIn*)) for the kernels'
// head dims too
template <typename F>
inline void for_type(int dtype, F&& fn) {
  if (dtype == HTREE_BF16)
    fn(std::integral_constant<bool, false>{}, (__bf16*)nullptr);
  else if (dtype == HTREE_F16)
    fn(std::integral_constant<bool, true>{}, (_Float16*)nullptr);
  else
    fn(std::integral_constant<bool, true>{}, (float*)nullptr);
}
template <typename F>
inline void for_dim_type(int D, int dtype, F&& fn) {
  auto by_type = [&](auto d) { for_type(dtype, [&](auto prec, auto* tin) { fn(d, prec, tin); }); };
  if (D == 256) by_type(std::integral_constant<int, 256>{});
  else if (D == 128) by_type(std::integral_constant<int, 128>{});
  else if (D == 32) by_type(std::integral_constant<int, 32>{});
  else by_type(std::integral_constant<int, 64>{});
}

}  // namespace htree
