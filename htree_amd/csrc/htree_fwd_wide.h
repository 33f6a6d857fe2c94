// Wide form of the fused forward (htree_fwd.hip describes the work the fused
// forwards share).  One source file per head dim instantiates it
// (htree_fwd_wide_d*.hip: the builds run side by side).
#pragma once

#include "htree_fwd.h"

namespace htree {

// ---------------------------------------------------------------- wide forward
// Levels of up to 16384 candidates (top_k up to 1024; the reference's default
// regime, src/parallel.py:537-867 with TOP_K = 512): one block of four waves
// per query group, in three steps per level.
//  1. Importance (upper levels): every tile scored once, tile tau by wave
//     tau mod 4, four tiles of the wave at a time, sum_g exp(s - m) per
//     position with m the wave's running max at the tile.  The four tiles'
//     maxima over the wave and their sums over the heads are reduced
//     together: two v_permlane16_swap and one v_permlane32_swap leave tile
//     j's partial in lane group j, where one tile by itself takes as many.
//     The arithmetic per tile (the query turned by the slot's table row, the
//     split products, m, the exponentials, the order of the sums) fixes which
//     nodes are selected and does not depend on this grouping.
//  2. Selection: a block-wide radix select over the float bits (BlockSelect);
//     thread i holds candidate positions Ci .. Ci+C-1 in registers (C = 32,
//     or 64 above 8192 positions), so ties at the threshold go to the lowest
//     positions (stable descending sort, src/naive.py:88-105).
//  3. Accumulation of the candidates not passed down: batches of four
//     consecutive tiles, rescored, one online-softmax step per batch
//     (a skipped rescale where no head's max rises).  The top level's
//     candidates are nodes 0 .. t's, met at R(K, node) with one turn of the
//     query; below, the query takes a batch's last slot from the table and
//     turns by CR per slot.
// Each wave keeps its own softmax state; they are merged at the end.
// D = 32 is bound by the vector data path (71% busy: 2.0 TB of operands a
// launch at T 120000, 64/4 heads, top_k 512) beside 58% of the vector ALU:
// 240 -> 133 ms there against one tile at a time, 24.0 -> 18.5 ms with 64 heads
// over one KV head at D = 64, 23.8 -> 10.2 ms at D = 128, T 16000, top_k 256
// (bf16).  Two waves per SIMD.  Split operands at D <= 64 spill there already
// (C = 32, 1 / 2 / 4 parts: D 32 fp32 24 / 29 / 43 VGPRs, D 64 fp32 35 / 42 /
// 45; bf16 4 to 11), which takes the same path: 12 GB written per launch at
// D = 32, 1 GB of it outputs.  At three waves more of the batches' operands
// spill and it is slower (165 ms).
// NH > 1 (kv_share 2 or 4: query groups of 17..32 or 33..64 heads): the
// block takes KV heads NH h' .. NH h' + NH - 1 of one query (their keys and
// values are the same), the kWideWaves / NH waves of part i the heads of KV
// head NH h' + i.  Each part keeps its own importance array and running
// maxima; the selection runs once, block-wide, over the parts' importance
// sum_i imp_i e^{m_i - M} (the group-shared sum over all of the group's
// heads), and every part takes its result.

// Reduces four values per lane (tile j in x_j) over the four lane groups:
// lane group j ends with op over the groups of x_j, (g0 op g1) op (g2 op g3).
template <typename Op>
__device__ __forceinline__ float groups4(float x0, float x1, float x2, float x3, Op op) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x0), __float_as_uint(x1), false, false);
  const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(x2), __float_as_uint(x3), false, false);
  const float u = op(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const float v = op(__uint_as_float(b[0]), __uint_as_float(b[1]));
  const auto c = __builtin_amdgcn_permlane32_swap(__float_as_uint(u), __float_as_uint(v), false, false);
  return op(__uint_as_float(c[0]), __uint_as_float(c[1]));
}
__device__ __forceinline__ float lane_f(float x, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
}

template <int D, bool PREC, typename TIn, bool TRACE, int C, int NH = 1, bool SEL = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D <= 128 && C == 32 ? 2 : 1))) void fwd_wide_kernel(const FwdArgs a) {
  static_assert(!(SEL && TRACE), "selection only: no trace");
  constexpr int KS = D / 32, ND = D / 16, HALF = D / 2;
  constexpr int U = kWideBatch;        // tiles of a batch: importance,
  constexpr int UA = D <= 64 ? 4 : 1;  // accumulation
  // D = 32: the next batch's keys (and the importance's table rows, through
  // LDS) are loaded while a batch is computed; D <= 64: a batch's values while
  // its tiles are scored.  The larger head dims have no registers for it
  // (D = 64 with the keys too: 300 spills, 16.7 against 17.0 ms).
  constexpr bool PIPE = D == 32;
  constexpr bool VPIPE = D <= 64;
  // P in bf16 hi + lo.  bf16 inputs at D <= 64 too: a batch's one softmax step
  // leaves fewer P that are exactly 1 than a step per tile (output error against
  // float64, D 32, T 4000: 1.96e-3 with a step per tile, 2.01e-3, and 1.62e-3
  // with P split).  A step per tile where some head's max rises, which more
  // than half of the batches see, cost more: T 8000, 64/4 heads, D 64 3.01 ->
  // 3.43 ms, P split 3.29.
  constexpr bool PSPLIT = PREC || UA > 1;
  static_assert(NH == 1 || NH == 2 || NH == 4, "parts of a block");
  // waves per part, threads
  constexpr int NW = kWideWaves / NH, NT = 64 * kWideWaves;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int part = NH > 1 ? wv / NW : 0, wvh = wv % NW;  // the wave's part, its wave within it
  const int u16 = lane & 15, kg = lane >> 4;
  const int G = a.G, CR = a.CR, crlg = a.crlg, TK = a.TK;
  const int CRU = CR < 16 ? CR : 16;
  const bool wide = CR >= 16;
  const int lgt = wide ? 4 : crlg;  // log2 of a tile's positions
  const WideLds LO = wide_lds(TK, TK << crlg, a.max_tiles, D, NH);
  int32_t* par = (int32_t*)(lds + LO.par);      // [2][TK]
  uint32_t* selw = (uint32_t*)(lds + LO.selw);  // selection bit of every position
  // running max of the wave at each tile (then its factor e^{m - M}),
  // importance of every position: per part
  float* mt0 = (float*)(lds + LO.mt);
  float* mt = mt0 + part * a.max_tiles;
  int32_t* red = (int32_t*)(lds + LO.red);      // [0,16) counts, [16,32) scans, [32,36) maxima
  float* imp0 = (float*)(lds + LO.imp);
  float* imp = imp0 + part * (TK << crlg);

  __shared__ __attribute__((aligned(16))) float tab[kWideWaves][PIPE ? wide_tab_floats(D) : 1];  // table rows of a batch

  const int64_t grp = (int64_t)(blockIdx.x & 7) * a.per_xcd + (blockIdx.x >> 3);
  if (grp >= (int64_t)a.B * a.Hkv * a.T / NH) return;  // uniform over the block
  int t, h, b;
  if (NH > 1) {  // block grp: query t of KV heads NH h' .. NH h' + NH - 1
    const int Hr = a.Hkv / NH;
    t = (int)(grp % a.T);
    const int64_t bhr = grp / a.T;
    h = NH * (int)(bhr % Hr) + part;
    b = (int)(bhr / Hr);
  } else {
    t = (int)(grp % a.T);
    const int bh = (int)(grp / a.T);
    h = bh % a.Hkv;
    b = bh / a.Hkv;
  }
  const int Gs = sel_heads(a, h);  // heads in the selection
  const bool gv = u16 < G;
  const int64_t hq = ((int64_t)b * a.T + t) * a.H + h * G + u16;
  // Rows past the group repeat its heads, so that their scores stay in the
  // range of the others (they are left out of the sums and not stored); a
  // padded group's are zero and masked to -inf, as its padding heads.
  const bool zero_row = !gv && a.gpad > 0;
  const TIn* qp = (const TIn*)a.q +
                  (((int64_t)b * a.T + t) * a.H + h * G + (gv ? u16 : a.gpad > 0 ? 0 : u16 % G)) * D;

  float m_run = -INFINITY, l_part = 0.f;
  f32x4 O[ND];
#pragma unroll
  for (int n = 0; n < ND; ++n) O[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  {
    const int64_t nvp = (t / a.lv[a.L - 1].pw) / CR + 1;  // src/naive.py:108-118
    for (int i = tid; i < TK; i += NT) par[i] = i < nvp ? i : -1;
  }

  // operand loads: a scalar tile address plus the lane's 32-bit offset
  const uint32_t koff = (u16 < CRU ? u16 : 0) * 16 + kg * 256;
  const uint32_t voff = (4 * kg < CRU ? 8 * D * kg : 0) + u16 * 16;
  auto load_k = [&](const uint16_t* base, int node0, bf16x8 (&f)[KS]) {
    const char* p = (const char*)(base + (int64_t)(node0 & ~15) * D + (node0 & 15) * 8);
#pragma unroll
    for (int m = 0; m < KS; ++m) f[m] = *(const bf16x8*)(p + m * 1024 + koff);
  };
  // V^T fragments of output tiles 2i, 2i + 1 (dims 32i + 2 u16, + 1): 16 bytes
  auto load_v = [&](const uint16_t* base, int node0, uint4 (&f)[ND / 2]) {
    const char* p = (const char*)(base + (int64_t)node0 * D);
#pragma unroll
    for (int i = 0; i < ND / 2; ++i) f[i] = *(const uint4*)(p + i * 256 + voff);
  };

  BlockSelect<C> bsel{red, lane, wv};
  // merge of a part's waves' states; the result (max, sum, output) is valid
  // in the part's first wave
  auto merge_waves = [&](float& Mo, float& Lo, f32x4 (&Om)[ND]) {
    const float lt = add_xor32(add_xor16(l_part));
    constexpr int DP = D + 1;
    float* mw = (float*)(lds + LO.imp + part * LO.merge_part);
    float* lw = mw + NW * 16;
    float* ow = mw + 2 * NW * 16;
    __syncthreads();
    if (kg == 0) {
      mw[wvh * 16 + u16] = m_run;
      lw[wvh * 16 + u16] = lt;
    }
#pragma unroll
    for (int n = 0; n < ND; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) ow[(wvh * 16 + u16) * DP + 16 * n + 4 * kg + r] = O[n][r];
    __syncthreads();
    if (wvh == 0) {
      float M = -INFINITY, L = 0.f;
#pragma unroll
      for (int n = 0; n < ND; ++n) Om[n] = f32x4{0.f, 0.f, 0.f, 0.f};
      for (int w = 0; w < NW; ++w) M = fmaxf(M, mw[w * 16 + u16]);
      if (M > -INFINITY) {
        for (int w = 0; w < NW; ++w) {
          const float mw_ = mw[w * 16 + u16];
          if (mw_ == -INFINITY) continue;
          const float sc = expf(mw_ - M);
          L += lw[w * 16 + u16] * sc;
#pragma unroll
          for (int n = 0; n < ND; ++n)
#pragma unroll
            for (int r = 0; r < 4; ++r) Om[n][r] += ow[(w * 16 + u16) * DP + 16 * n + 4 * kg + r] * sc;
        }
      }
      Mo = M;
      Lo = L;
    }
  };

  int cur = 0;
  for (int l = a.L - 1; l >= 0; --l) {
    __syncthreads();
    const LevelPtrs P = a.lv[l];
    const int32_t* pc = par + cur * TK;
    int lo = 0, hi = TK;  // the valid entries are a prefix of the list
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (pc[mid] >= 0) lo = mid + 1; else hi = mid;
    }
    const int np = uniform(lo);
    const int ct = uniform((int)((t / P.pw) & (CR - 1)));
    const int nc = ((np - 1) << crlg) + ct + 1;
    const int apos = nc - 1;
    const int nt = wide ? (nc + 15) >> 4 : np;
    if (a.parents)  // (each part its own head's row)
      for (int i = tid - part * 64 * NW; i < TK; i += 64 * NW)
        a.parents[((((int64_t)l * a.B + b) * a.T + t) * a.Hkv + h) * TK + i] = pc[i];
    if (SEL && l == 0) break;  // the bottom level selects nothing (uniform over the block)
    const int64_t hrow = ((int64_t)b * a.Hkv + h) * P.Np;
    const bool top = l == a.L - 1;
    const bool upper = l > 0;
    auto slot_of = [&](int tau) { return wide ? (tau << 4) >> crlg : tau; };
    auto node0_of = [&](int tau) {  // (the same in every lane: scalar addresses)
      return (uniform(pc[slot_of(tau)]) << crlg) + (wide ? ((tau << 4) & (CR - 1)) : 0);
    };

    // a level of at most top_k candidates passes all of them down: no scores,
    // nothing accumulated (src/naive.py:97-101)
    if (upper && nc <= TK) {
      int32_t* pn = par + (cur ^ 1) * TK;
      for (int i = tid; i < TK; i += NT)
        pn[i] = i < nc ? (pc[i >> crlg] << crlg) + (i & (CR - 1)) : -1;
      if (TRACE && wvh == 0) {
        f32x4 z[ND];
#pragma unroll
        for (int n = 0; n < ND; ++n) z[n] = f32x4{0.f, 0.f, 0.f, 0.f};
        trace_store<D>(a, l, hq, gv, kg, -INFINITY, 0.f, z);
      }
      cur ^= 1;
      continue;
    }
    if (upper) {
      // ---- importance of every candidate (relative to the wave's running max)
      const uint16_t* KH = P.sh + hrow * D;
      const uint16_t* KL = P.sl + hrow * D;
      // rows past the heads of the selection repeat them: no row's score is
      // out of the range of the others
      const TIn* qs = (const TIn*)a.q +
                      (((int64_t)b * a.T + t) * a.H + h * G + (u16 < Gs ? u16 : u16 % Gs)) * D;
      float qf[KS][8], qo[8];
#pragma unroll
      for (int m = 0; m < KS; ++m) {
        Io<TIn>::ld8(qs + dslot<D>(kg, m), qf[m]);
#pragma unroll
        for (int e = 0; e < 8; ++e) qf[m][e] *= a.scale;
      }
      if constexpr (D == 32) {  // the other halves of the lane's pairs, signed for the turn
        Io<TIn>::ld8(qs + (dslot<D>(kg, 0) ^ 16), qo);
#pragma unroll
        for (int e = 0; e < 8; ++e) qo[e] *= kg < 2 ? -a.scale : a.scale;
      }
      float hm[4];  // 1 for heads of the selection
#pragma unroll
      for (int r = 0; r < 4; ++r) hm[r] = 4 * kg + r < Gs ? 1.f : 0.f;
      float Mrun = -INFINITY;
      auto tile_at = [&](int i0, int j) { return i0 + NW * j < nt ? i0 + NW * j : nt - 1; };
      auto row_at = [&](int i0, int j) { return apos - (slot_of(tile_at(i0, j)) << crlg); };
      bf16x8 kh[U][KS], kl[U][KS];
      auto keys = [&](int i0) {
#pragma unroll
        for (int j = 0; j < U; ++j) {
          const int node0 = node0_of(tile_at(i0, j));
          load_k(KH, node0, kh[j]);
          load_k(KL, node0, kl[j]);
        }
      };
      // the batch's four table rows, cos then sin, an element of each lane
      float tb[U * D / 64];
      auto rows = [&](int i0) {
#pragma unroll
        for (int k = 0; k < U * D / 64; ++k) {
          const int w = (lane + 64 * k) % D;
          tb[k] = (w < HALF ? a.cosb : a.sinb - HALF)[(int64_t)row_at(i0, (lane + 64 * k) / D) * HALF + w];
        }
      };
      float* tabw = tab[wv];
      if (PIPE && wvh < nt) {
        rows(wvh);
        keys(wvh);
      }
      for (int i0 = wvh; i0 < nt; i0 += U * NW) {
        f32x4 S[U];
        if constexpr (PIPE) {
#pragma unroll
          for (int k = 0; k < U * D / 64; ++k) tabw[lane + 64 * k] = tb[k];
          wave_sync();
          rows(i0 + U * NW < nt ? i0 + U * NW : i0);
        }
#pragma unroll
        for (int j = 0; j < U; ++j) {
          float qr[KS][8];
          const int prow = row_at(i0, j);
          const float* cr = PIPE ? tabw + D * j : a.cosb + (int64_t)prow * HALF;
          const float* sr = PIPE ? tabw + D * j + HALF : a.sinb + (int64_t)prow * HALF;
          if constexpr (D == 32) {
            float c[8], s[8];
            Io<float>::ld8(cr + 8 * (kg & 1), c);
            Io<float>::ld8(sr + 8 * (kg & 1), s);
#pragma unroll
            for (int e = 0; e < 8; ++e) qr[0][e] = qf[0][e] * c[e] + qo[e] * s[e];
          } else {
            rope_frag<D>(qf, cr, sr, kg, qr);
          }
          bf16x8 qh[KS], ql[KS];
          to_bf_split<D>(qr, qh, ql);
          if (!PIPE) {
            const int node0 = node0_of(tile_at(i0, j));
            load_k(KH, node0, kh[j]);
            load_k(KL, node0, kl[j]);
          }
          S[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int m = 0; m < KS; ++m) {
            S[j] = mma32(qh[m], kh[j][m], S[j]);
            S[j] = mma32(qh[m], kl[j][m], S[j]);
            S[j] = mma32(ql[m], kh[j][m], S[j]);
          }
          if (!PIPE) __builtin_amdgcn_sched_barrier(0);  // one tile's keys in registers
        }
        if (PIPE) keys(i0 + U * NW < nt ? i0 + U * NW : i0);
        // S[j][r] = score[g = 4kg + r][candidate u16 of tile i0 + NW j].  A
        // column that is no candidate is kept out of the max and its sum not
        // stored; its scores (of some node of the tree) stay as they are, so
        // that the subnormal test below sees no -inf
        float tm[U], M[U];
#pragma unroll
        for (int j = 0; j < U; ++j) tm[j] = fmaxf(fmaxf(S[j][0], S[j][1]), fmaxf(S[j][2], S[j][3]));
        if (!wide || i0 + NW * (U - 1) >= nt - 1) {
#pragma unroll
          for (int j = 0; j < U; ++j) {
            const int tau = i0 + NW * j;
            const bool cv = tau < nt && u16 < CRU && (tau << lgt) + u16 < nc;
            tm[j] = cv ? tm[j] : -INFINITY;
          }
        }
        const float tmx = row_max16(groups4(tm[0], tm[1], tm[2], tm[3], [](float x, float y) { return fmaxf(x, y); }));
#pragma unroll
        for (int j = 0; j < U; ++j) {
          Mrun = fmaxf(Mrun, lane_f(tmx, 16 * j));
          M[j] = Mrun;
        }
        float xm = 0.f;
#pragma unroll
        for (int j = 0; j < U; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            S[j][r] = (S[j][r] - M[j]) * kLog2e;
            xm = fminf(xm, S[j][r]);
          }
        float e[U];
        if (__builtin_expect(__any(xm < -126.f), 0)) {  // subnormal results (exp_sel)
#pragma unroll
          for (int j = 0; j < U; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const bool sb = S[j][r] < -126.f;
              const float p = __builtin_amdgcn_exp2f(sb ? S[j][r] + 64.f : S[j][r]);
              S[j][r] = sb ? p * 5.42101086242752217e-20f : p;
            }
        } else {
#pragma unroll
          for (int j = 0; j < U; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) S[j][r] = __builtin_amdgcn_exp2f(S[j][r]);
        }
#pragma unroll
        for (int j = 0; j < U; ++j) {
          e[j] = 0.f;
#pragma unroll
          for (int r = 0; r < 4; ++r) e[j] = fmaf(S[j][r], hm[r], e[j]);
        }
        const float es = groups4(e[0], e[1], e[2], e[3], [](float x, float y) { return x + y; });
        const int tk = i0 + NW * kg;  // this lane group's tile
        const int pos = (tk << lgt) + u16;
        if (tk < nt && u16 < CRU && pos < nc) imp[pos] = es;
        if (u16 == 0 && tk < nt) mt[tk] = kg < 2 ? (kg == 0 ? M[0] : M[1]) : (kg == 2 ? M[2] : M[3]);
      }
      if (lane == 0) red[32 + wv] = __float_as_int(Mrun);
      __syncthreads();
      const float M = fmaxf(fmaxf(__int_as_float(red[32]), __int_as_float(red[33])),
                            fmaxf(__int_as_float(red[34]), __int_as_float(red[35])));
      for (int i = tid; i < NH * a.max_tiles; i += NT)
        if (i % a.max_tiles < nt) mt0[i] = mt0[i] != M ? expf(mt0[i] - M) : 1.f;
      __syncthreads();
      // ---- keys: float bits + 1 (0 = no candidate); rightmost forced (src/naive.py:93)
      const int take = TK < nc ? TK : nc;
      // (an opaque copy: the positions' offsets are formed here, not hoisted
      // out of the level loop and held through the scoring loops)
      int tq = tid;
      asm volatile("" : "+v"(tq));
      uint32_t key[C];
#pragma unroll
      for (int i = 0; i < C; ++i) key[i] = 0u;
      bsel.has = wv * 64 * C < nc;
      if (tq * C < nc) {
#pragma unroll
        for (int i4 = 0; i4 < C; i4 += 4) {
#pragma clang fp contract(off)  // each part's sum is rounded before it is added
          float v[4];
#pragma unroll
          for (int j = 0; j < NH; ++j) {  // the parts' sums, in a fixed order
            const float4 x = *(const float4*)(imp0 + j * (TK << crlg) + tq * C + i4);
            const float xv[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {  // (four positions lie in one tile)
              const float f = xv[i] * mt0[j * a.max_tiles + ((tq * C + i4) >> lgt)];
              v[i] = j == 0 ? f : v[i] + f;
            }
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int pos = tq * C + i4 + i;
            if (pos < nc) key[i4 + i] = __float_as_uint(pos == apos ? 1e6f : v[i]) + 1u;
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      // ---- the take-th largest key, bit by bit from the top (keys < 2^31)
      int idx;
      const auto bits = bsel.select(key, take, 30, idx);
      int32_t* pn = par + (cur ^ 1) * TK;
      for (auto bb = bits; bb != 0; bb &= bb - 1) {
        const int pos = tq * C + __builtin_ctzll((unsigned long long)bb);
        pn[idx++] = (pc[pos >> crlg] << crlg) + (pos & (CR - 1));
      }
      if (tq * C < (TK << crlg)) {
        selw[tq * (C / 32)] = (uint32_t)bits;
        if constexpr (C == 64) selw[tq * 2 + 1] = (uint32_t)((unsigned long long)bits >> 32);
      }
      for (int i = take + tq; i < TK; i += NT) pn[i] = -1;
      __syncthreads();
    }
    if constexpr (SEL) {
      cur ^= 1;
      continue;
    }

    // ---- accumulation of the candidates not passed down
    if (TRACE) {
      m_run = -INFINITY;
      l_part = 0.f;
#pragma unroll
      for (int n = 0; n < ND; ++n) O[n] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const uint16_t* KH = P.kh + hrow * D;  // (the top level's at the angle of the node)
    const uint16_t* KL = P.kl + hrow * D;
    const uint16_t* VH = P.vh + hrow * D;
    const uint16_t* VL = PREC ? P.vl + hrow * D : nullptr;
    float qf[KS][8];
#pragma unroll
    for (int m = 0; m < KS; ++m) {
      ld_pairs<D, TIn>(qp, kg, m, qf[m]);
#pragma unroll
      for (int e = 0; e < 8; ++e) qf[m][e] = zero_row ? 0.f : qf[m][e] * a.scale;
    }
    bf16x8 qh[KS], ql[KS];
    if (top) {
      float qr[KS][8];
      rope_frag<D>(qf, a.cosb + (int64_t)apos * HALF, a.sinb + (int64_t)apos * HALF, kg, qr);
      to_bf_split<D>(qr, qh, ql);
    }
    const int nb = (nt + UA - 1) / UA;
    // The batches of a level.  FORM 0: the top level of a tree (whole tiles of
    // 16, one query frame, candidates passed down masked); 1: the bottom
    // level, a slot per tile; 2: any level (the branches stay in the loop).
    auto accumulate = [&](auto form) __attribute__((always_inline)) {
      constexpr int FORM = decltype(form)::value;
      const bool masks = FORM == 0 || (FORM == 2 && upper);
      const bool one_frame = FORM == 0 || (FORM == 2 && top);
      // tiles of fewer than 16 candidates: the lane groups past them start at -inf
      const float c0 = FORM == 2 && 4 * kg >= CRU ? -INFINITY : 0.f;
      const float* ccr = a.cosb + (int64_t)CR * HALF;  // the angle CR
      const float* scr = a.sinb + (int64_t)CR * HALF;
      auto nodes = [&](int bi, int (&nd)[UA]) {
        const int tau0 = bi * UA;
        if constexpr (FORM == 0) {
#pragma unroll
          for (int j = 0; j < UA; ++j) nd[j] = 16 * (tau0 + j < nt ? tau0 + j : nt - 1);
        } else if constexpr (FORM == 1) {  // (entries past the list are -1)
#pragma unroll
          for (int j = 0; j < UA; ++j) nd[j] = max(uniform(pc[tau0 + j]), 0) << crlg;
        } else {
#pragma unroll
          for (int j = 0; j < UA; ++j) nd[j] = node0_of(tau0 + j < nt ? tau0 + j : nt - 1);
        }
      };
      bf16x8 kh[UA][KS], kl[UA][KS];
      auto keys = [&](const int (&nd)[UA]) {
#pragma unroll
        for (int j = 0; j < UA; ++j) {
          load_k(KH, nd[j], kh[j]);
          load_k(KL, nd[j], kl[j]);
        }
      };
      int nd[UA];
      if (wvh < nb) nodes(wvh, nd);
      if (PIPE && wvh < nb) keys(nd);
      for (int bi = wvh; bi < nb; bi += NW) {
        const int tau0 = bi * UA;
        const bool last = bi == nb - 1;
        f32x4 S[UA];
        uint4 vh[UA][ND / 2], vl[UA][ND / 2];
        if (VPIPE) {  // in flight while the tiles are scored
#pragma unroll
          for (int j = 0; j < UA; ++j) {
            load_v(VH, nd[j], vh[j]);
            if (PREC) load_v(VL, nd[j], vl[j]);
          }
        }
        // tiles in descending slot: the query turns on by CR per slot
        float qr[KS][8];
        int cs = -1;
#pragma unroll
        for (int j = UA - 1; j >= 0; --j) {
          const int tau = tau0 + j < nt ? tau0 + j : nt - 1;
          if (!one_frame) {
            const int s = FORM == 1 ? tau0 + j : slot_of(tau);
            // (D >= 128, batches of one tile: from the table at every slot, as
            // turning on would hold the query twice and the angle's row in registers)
            if (j == UA - 1) {
              const int prow = apos - (s << crlg);
              if (FORM == 1 && prow < 0) {
                // a slot past the list (the last batch turns back from it):
                // R(q, -p) turns the conjugate pairs by p
                float qc[KS][8];
                auto conj = [&](const float (&x)[KS][8], float (&y)[KS][8]) {
#pragma unroll
                  for (int m = 0; m < KS; ++m)
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                      const bool hi = D == 32 ? e >= 4 : m >= KS / 2;
                      y[m][e] = hi ? -x[m][e] : x[m][e];
                    }
                };
                conj(qf, qc);
                rope_frag<D>(qc, a.cosb - (int64_t)prow * HALF, a.sinb - (int64_t)prow * HALF, kg, qr);
                conj(qr, qr);
              } else {
                rope_frag<D>(qf, a.cosb + (int64_t)prow * HALF, a.sinb + (int64_t)prow * HALF, kg, qr);
              }
              to_bf_split<D>(qr, qh, ql);
            } else if (FORM == 1 || s != cs) {
              rope_frag<D>(qr, ccr, scr, kg, qr);
              to_bf_split<D>(qr, qh, ql);
            }
            cs = s;
          }
          if (!PIPE) {
            load_k(KH, nd[j], kh[j]);
            load_k(KL, nd[j], kl[j]);
          }
          f32x4 ci = {c0, c0, c0, c0};
          if (masks) {  // -inf where the candidate is passed down
            const int p0 = tau << lgt;
            const uint32_t w = (uint32_t)uniform((int)selw[p0 >> 5]) >> (p0 & 31);
#pragma unroll
            for (int r = 0; r < 4; ++r)
              ci[r] = __int_as_float((__builtin_amdgcn_sbfe((int)w, 4 * kg + r, 1) & 0xff800000) |
                                     (FORM == 2 ? __float_as_int(c0) : 0));
          }
          S[j] = ci;
#pragma unroll
          for (int m = 0; m < KS; ++m) {
            S[j] = mma32(kh[j][m], qh[m], S[j]);
            S[j] = mma32(kl[j][m], qh[m], S[j]);
            S[j] = mma32(kh[j][m], ql[m], S[j]);
          }
          if (!PIPE) __builtin_amdgcn_sched_barrier(0);
        }
        int nn[UA];
        nodes(last || bi + NW >= nb ? bi : bi + NW, nn);
        if (PIPE) keys(nn);
        // S[j][r] = score[candidate 4kg + r of tile tau0 + j][g = u16]
        if (last) {
#pragma unroll
          for (int j = 0; j < UA; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const bool ok = tau0 + j < nt && ((tau0 + j) << lgt) + 4 * kg + r < nc;
              S[j][r] = ok ? S[j][r] : -INFINITY;
            }
        }
        float tm = S[0][0];
#pragma unroll
        for (int j = 0; j < UA; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) tm = fmaxf(tm, S[j][r]);
        tm = max_xor32(max_xor16(tm));
        if (__any(tm > m_run)) {
          const float mnew = fmaxf(m_run, tm);
          const float alpha = mnew == -INFINITY ? 1.f : __builtin_amdgcn_exp2f((m_run - mnew) * kLog2e);
          m_run = mnew;
          l_part *= alpha;
#pragma unroll
          for (int n = 0; n < ND; ++n) O[n] *= alpha;
        }
        const float mref = m_run == -INFINITY ? 0.f : m_run;
#pragma unroll
        for (int j = 0; j < UA; ++j) {
          if (!VPIPE) {
            load_v(VH, nd[j], vh[j]);
            if (PREC) load_v(VL, nd[j], vl[j]);
          }
          float p[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) p[r] = __builtin_amdgcn_exp2f((S[j][r] - mref) * kLog2e);
          l_part += (p[0] + p[1]) + (p[2] + p[3]);
          const uint32_t h01 = cvt_pk_bf16(p[0], p[1]), h23 = cvt_pk_bf16(p[2], p[3]);
          const s16x4 ph = __builtin_bit_cast(s16x4, make_uint2(h01, h23));
          s16x4 pl = ph;
          if (PSPLIT) {
            const uint32_t l01 = cvt_pk_bf16(p[0] - __uint_as_float(h01 << 16),
                                             p[1] - __uint_as_float(h01 & 0xffff0000u));
            const uint32_t l23 = cvt_pk_bf16(p[2] - __uint_as_float(h23 << 16),
                                             p[3] - __uint_as_float(h23 & 0xffff0000u));
            pl = __builtin_bit_cast(s16x4, make_uint2(l01, l23));
          }
#pragma unroll
          for (int i = 0; i < ND / 2; ++i) {
            const uint4 w = vh[j][i];
            const s16x4 v0 = __builtin_bit_cast(s16x4, make_uint2(w.x, w.y));
            const s16x4 v1 = __builtin_bit_cast(s16x4, make_uint2(w.z, w.w));
            O[2 * i] = mma16(v0, ph, O[2 * i]);
            O[2 * i + 1] = mma16(v1, ph, O[2 * i + 1]);
            if (PSPLIT) {
              O[2 * i] = mma16(v0, pl, O[2 * i]);
              O[2 * i + 1] = mma16(v1, pl, O[2 * i + 1]);
            }
            if (PREC) {
              const uint4 wl = vl[j][i];
              const s16x4 l0 = __builtin_bit_cast(s16x4, make_uint2(wl.x, wl.y));
              const s16x4 l1 = __builtin_bit_cast(s16x4, make_uint2(wl.z, wl.w));
              O[2 * i] = mma16(l0, ph, O[2 * i]);
              O[2 * i + 1] = mma16(l1, ph, O[2 * i + 1]);
            }
          }
        }
#pragma unroll
        for (int j = 0; j < UA; ++j) nd[j] = nn[j];
      }
    };
    if (D <= 64 && top && upper && wide)
      accumulate(std::integral_constant<int, D <= 64 ? 0 : 2>{});
    else if (D <= 64 && !upper && !top && CR == 16 && TK >= UA)
      accumulate(std::integral_constant<int, D <= 64 ? 1 : 2>{});
    else
      accumulate(std::integral_constant<int, 2>{});
    if (TRACE) {
      float Ml, Ll;
      f32x4 Ol[ND];
      merge_waves(Ml, Ll, Ol);
      if (wvh == 0) trace_store<D>(a, l, hq, gv, kg, Ml, kg == 0 ? Ll : 0.f, Ol);
    }
    cur ^= 1;
  }

  if constexpr (SEL) return;
  float M, lt;
  if (TRACE) {
    if (wvh != 0) return;
    lt = trace_merge<D>(a, hq, gv, kg, M, O);
  } else {
    merge_waves(M, lt, O);
    if (wvh != 0) return;
  }
  if (gv) {
    const float inv = 1.f / lt;
    store_out<D, TIn>((TIn*)a.out + hq * D, kg, O, [&](float x) { return x * inv; });
    if (kg == 0) {
      a.gmax[hq] = M;
      a.gsum[hq] = lt;
    }
  }
}

// the wide forward with NH parts per block (kv_share 1, 2 or 4); sel: the
// selection-only instances
template <int D, bool PREC, typename TIn, int NH>
static void launch_wide(const FwdArgs& a, dim3 grid, hipStream_t st, bool sel) {
  const unsigned lds = (unsigned)wide_lds(a.TK, a.TK << a.crlg, a.max_tiles, D, NH).bytes;
  const bool c64 = (a.TK << a.crlg) > kWideMidPos;  // 64 keys per thread
  if (sel) {
    if (c64)
      hipLaunchKernelGGL((fwd_wide_kernel<D, PREC, TIn, false, 64, NH, true>), grid, dim3(256), lds, st, a);
    else
      hipLaunchKernelGGL((fwd_wide_kernel<D, PREC, TIn, false, 32, NH, true>), grid, dim3(256), lds, st, a);
  } else if (a.tout != nullptr) {
    if (c64)
      hipLaunchKernelGGL((fwd_wide_kernel<D, PREC, TIn, true, 64, NH>), grid, dim3(256), lds, st, a);
    else
      hipLaunchKernelGGL((fwd_wide_kernel<D, PREC, TIn, true, 32, NH>), grid, dim3(256), lds, st, a);
  } else {
    if (c64)
      hipLaunchKernelGGL((fwd_wide_kernel<D, PREC, TIn, false, 64, NH>), grid, dim3(256), lds, st, a);
    else
      hipLaunchKernelGGL((fwd_wide_kernel<D, PREC, TIn, false, 32, NH>), grid, dim3(256), lds, st, a);
  }
}

template <int D>
void launch_fwd_wide_d(int dtype, const FwdArgs& a, dim3 grid, hipStream_t st, bool sel) {
  for_type(dtype, [&](auto prec, auto* tin) {
    using TIn = typename std::remove_pointer<decltype(tin)>::type;
    constexpr bool PREC = decltype(prec)::value;
    if (a.kv_share == 4)  // one block per four KV heads of a query (any level size)
      launch_wide<D, PREC, TIn, 4>(a, grid, st, sel);
    else if (a.kv_share == 2)  // one block per KV-head pair of a query
      launch_wide<D, PREC, TIn, 2>(a, grid, st, sel);
    else  // one block per query group
      launch_wide<D, PREC, TIn, 1>(a, grid, st, sel);
  });
}

}  // namespace htree
