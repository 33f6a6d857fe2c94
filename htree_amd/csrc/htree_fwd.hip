// Fused htree forward: one wave per query group (b, t, h_kv) walks every
// tree level top -> bottom with its online-softmax state in registers.
//
// Reference behaviour (file:line in /root/reference):
//   candidate expansion, rightmost truncation ...... src/naive.py:180-191,
//                                                    src/parallel.py:409-426
//   RoPE on q at n_c-1 and on k at the flat position src/naive.py:193-199
//   group-shared importance, forced rightmost,
//   stable top-k (lower position wins ties) ....... src/naive.py:88-105,201-207,
//                                                    src/parallel.py:721-771
//   online softmax of the non-selected candidates . src/naive.py:73-85,209-213
//   cross-level merge, out = o / s ................. src/naive.py:215-231,
//                                                    src/parallel.py:248-363
//
// Layout of the work (gfx950, wave64, MFMA 16x16):
//   candidates are processed in tiles of 16 consecutive children of one
//   parent (one tile per parent when CR < 16).  RoPE uses angle addition:
//   R(q, a) . R(k, j) = R(q, a - s*CR) . R(k, j mod CR) for j in parent slot
//   s, so K is stored pre-rotated by its node's child index and the query is
//   rotated once per tile.
//   Scores use a split-bf16 product (qh*kh + qh*kl + ql*kh, error ~1e-5 of
//   |q||k| scale); P.V uses plain bf16 for bf16 inputs (V exact, P rounded)
//   and the split product for fp32/fp16 inputs.
//   O is accumulated transposed (O^T = V^T P^T) so that each lane owns one
//   query head and the softmax rescale needs no cross-lane traffic.
#include <string.h>

#include "htree_fwd.h"

namespace htree {

// Shared Top-K of the group (src/naive.py:88-105): importance of position j
// is imp[j] (lane j % 64 of slot j / 64), the rightmost (position apos) is
// forced first; a bitwise radix select on float bits + 1 finds the take-th
// largest key (16 steps, then 15 more only when the keys sharing its top 16
// bits do not settle it), ties at the threshold go to the lowest positions
// (stable descending sort).  Writes the selected nodes in ascending order
// (= ascending position) to par_next, -1 padded to TK, and one selection
// bitmask per slot to selmask.
// With imp2 (a pair of KV heads sharing the selection), the importance of
// position j is imp[j] f1 + imp2[j] f2: each array is relative to its own
// half's level max, f = exp(m_half - m_pair); both waves of the pair pass
// the arrays in the same order, so both select the same nodes.
template <int MAXSLOT>
__device__ __forceinline__ void select_topk(const float* __restrict__ imp, int nt, int nc, int apos,
                                            int TK, bool wide, int crlg, int CR, int CRU,
                                            const int32_t* par_cur, int32_t* par_next,
                                            unsigned long long* selmask, int lane,
                                            const float* __restrict__ imp2 = nullptr,
                                            float f1 = 1.f, float f2 = 0.f) {
  const int u16 = lane & 15, kg = lane >> 4;
  const int take = uniform(TK < nc ? TK : nc);
  const int nslot = uniform((nt + 3) >> 2);
  uint32_t key[MAXSLOT];
#pragma unroll
  for (int sl = 0; sl < MAXSLOT; ++sl) {
    key[sl] = 0u;
    if (sl < nslot) {
      const int tau = 4 * sl + kg;
      const int pos = wide ? (tau << 4) + u16 : (tau << crlg) + u16;
      if (tau < nt && u16 < CRU && pos < nc) {
        float v;
        if (pos == apos) {
          v = 1e6f;  // rightmost candidate always kept (src/naive.py:93)
        } else {
          v = imp2 ? imp[64 * sl + lane] * f1 + imp2[64 * sl + lane] * f2 : imp[64 * sl + lane];
        }
        key[sl] = __float_as_uint(v) + 1u;
      }
    }
  }
  // The take-th largest key, bit by bit from the top.  The keys of the
  // slots past nslot are 0 and never counted (c >= 1), so up to four slots
  // are counted unconditionally.
  auto radix = [&](uint32_t thr, int hi, int lo) {
    for (int bit = hi; bit >= lo; --bit) {
      const uint32_t c = thr | (1u << bit);
      int cnt = 0;
#pragma unroll
      for (int sl = 0; sl < MAXSLOT; ++sl)
        if (MAXSLOT <= 4 || sl < nslot) cnt += __popcll(__ballot(key[sl] >= c));
      if (cnt >= take) thr = c;
    }
    return thr;
  };
  // bits 30..15 first; the keys that share them hold the take-th largest,
  // which is their largest when one more is needed, their smallest when all
  // of them are, the common value when they are equal, else bits 14..0
  uint32_t thr = radix(0u, 30, 15);
  {
    int above = 0, neq = 0;
    float emax = 0.f, emin = -INFINITY;  // keys read as floats keep their order
#pragma unroll
    for (int sl = 0; sl < MAXSLOT; ++sl) {
      if (MAXSLOT <= 4 || sl < nslot) {
        const bool in = (key[sl] >> 15) == (thr >> 15);
        above += __popcll(__ballot((key[sl] >> 15) > (thr >> 15)));
        neq += __popcll(__ballot(in));
        if (in) {
          emax = fmaxf(emax, __uint_as_float(key[sl]));
          emin = fmaxf(emin, -__uint_as_float(key[sl]));
        }
      }
    }
    const int need2 = take - above;  // 1 <= need2 <= neq
    const uint32_t kmax = __float_as_uint(wave_max_uniform(emax));
    const uint32_t kmin = __float_as_uint(-wave_max_uniform(emin));
    if (need2 == 1 || kmin == kmax)
      thr = kmax;
    else if (need2 == neq)
      thr = kmin;
    else
      thr = radix(thr, 14, 0);
  }
  int ngt = 0;
#pragma unroll
  for (int sl = 0; sl < MAXSLOT; ++sl)
    if (MAXSLOT <= 4 || sl < nslot) ngt += __popcll(__ballot(key[sl] > thr));
  const int need = take - ngt;
  int eq_before = 0, sel_before = 0;
#pragma unroll
  for (int sl = 0; sl < MAXSLOT; ++sl) {
    if (sl < nslot) {
      const unsigned long long em = __ballot(key[sl] == thr);
      const bool sel = key[sl] > thr || (key[sl] == thr && eq_before + mbcnt64(em) < need);
      const unsigned long long sm = __ballot(sel);
      if (lane == 0) selmask[sl] = sm;
      if (sel) {
        const int tau = 4 * sl + kg;
        const int s = wide ? (tau << 4) >> crlg : tau;
        par_next[sel_before + mbcnt64(sm)] =
            (par_cur[s] << crlg) + (wide ? ((tau << 4) & (CR - 1)) : 0) + u16;
      }
      eq_before += __popcll(em);
      sel_before += __popcll(sm);
    }
  }
  if (lane >= take && lane < TK) par_next[lane] = -1;
}

// ---------------------------------------------------------------- single-pass forward
// For levels of at most 16 candidate tiles (TK * max(CR,16) <= 256): every
// tile is scored once (S^T, candidates x heads) into LDS; the selection uses
// the exact level max and the accumulation reuses the scores.  Tiles are
// walked in descending parent slot, so the query rotation advances by the
// constant angle CR (R(q, a - s CR) = R(R(q, a - (s+1) CR), CR)).  The V
// gathers are double-buffered one tile ahead; the K gathers are not (a
// second K buffer spills registers at two waves per SIMD, which costs more
// than it hides).
struct WaveLdsR {
  f32x4 st[16][64];  // S^T of every tile, one f32x4 per lane
  int32_t par[2][kMaxTK];
  float imp[256];
  unsigned long long selmask[4];
  float lvl_max;     // the level's max score of this wave's heads (KV-head pairs)
};

// SEL: selection only (the reference's htree_recompute_selection_kernel,
// src/parallel.py:1168): the parent lists of every level, no accumulation
// and no output.
template <int D, bool PREC, typename TIn, bool TRACE, bool SEL = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D == 256 ? 1 : 2))) void fwd_reg_kernel(const FwdArgs a) {
  static_assert(!(SEL && TRACE), "selection only: no trace");
  constexpr int KS = D / 32, ND = D / 16, HALF = D / 2;
  __shared__ WaveLdsR lds_all[kWavesPerBlock];
  __shared__ float rot_cr[2][HALF];  // cos / sin of the angle CR

  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int u16 = lane & 15, kg = lane >> 4;
  const int G = a.G, CR = a.CR, crlg = a.crlg, TK = a.TK;
  if (threadIdx.x < HALF) {
    rot_cr[0][threadIdx.x] = a.cosb[(int64_t)CR * HALF + threadIdx.x];
    rot_cr[1][threadIdx.x] = a.sinb[(int64_t)CR * HALF + threadIdx.x];
  }
  __syncthreads();
  const int bid = blockIdx.x;
  const int64_t lb = (int64_t)(bid & 7) * a.per_xcd + (bid >> 3);
  const int64_t grp = lb * kWavesPerBlock + wv;
  // A top level of <= top_k nodes keeps every candidate and accumulates
  // none (src/naive.py:97-101): its list is the virtual parents and its
  // selection every top node up to t's, so the walk starts one level lower.
  const bool skip_top = !TRACE && a.L > 1 && a.lv[a.L - 1].N <= TK;
  const int lstart = skip_top ? a.L - 2 : a.L - 1;
  // KV-head pairs (kv_share 2): waves 2i and 2i+1 of a block take KV heads
  // 2h, 2h+1 of one query and meet at two block barriers per upper level to
  // combine their importances.  Pairs never straddle blocks (the group count
  // is even), and the waves of an empty pair still pass every barrier.
  const bool pair = a.kv_share == 2;
  if (grp >= (int64_t)a.B * a.Hkv * a.T) {
    if (pair)
      for (int l = lstart; l >= 1; --l) {
        __syncthreads();
        __syncthreads();
      }
    return;
  }
  int t, h, b;
  if (pair) {
    const int Hr = a.Hkv >> 1;
    const int64_t pq = grp >> 1;
    t = (int)(pq % a.T);
    const int64_t bhr = pq / a.T;
    h = 2 * (int)(bhr % Hr) + (int)(grp & 1);
    b = (int)(bhr / Hr);
  } else {
    t = (int)(grp % a.T);
    const int bh = (int)(grp / a.T);
    h = bh % a.Hkv;
    b = bh / a.Hkv;
  }
  WaveLdsR& W = lds_all[wv];
  const int CRU = CR < 16 ? CR : 16;
  const bool wide = CR >= 16;
  const bool gv = u16 < G;

  // the query stays in its input type (16-bit types packed: 16 registers)
  QFrag<D, TIn, false> qin;
  // rows past the group repeat its heads: their scores stay in the range of
  // the others, and they are left out of the sums (hv) and not stored
  qin.load((const TIn*)a.q + (((int64_t)b * a.T + t) * a.H + h * G + (gv ? u16 : u16 % G)) * D, kg, true);
  const float hv = gv ? 1.f : 0.f;

  float m_run = -INFINITY, l_part = 0.f;
  f32x4 O[ND];
#pragma unroll
  for (int n = 0; n < ND; ++n) O[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  {
    const int64_t nvp = (t / a.lv[a.L - 1].pw) / CR + 1;
    if (lane < TK) W.par[0][lane] = lane < nvp ? lane : -1;
    if (skip_top) {
      if (a.parents && lane < TK)
        a.parents[((((int64_t)(a.L - 1) * a.B + b) * a.T + t) * a.Hkv + h) * TK + lane] =
            lane < nvp ? lane : -1;
      const int64_t ntop = t / a.lv[a.L - 1].pw + 1;
      if (lane < TK) W.par[0][lane] = lane < ntop ? lane : -1;
    }
  }
  int cur = 0;

  for (int l = lstart; l >= 0; --l) {
    wave_sync();
    const LevelPtrs P = a.lv[l];
    const int pv = lane < TK ? W.par[cur][lane] : -1;
    const int np = __popcll(__ballot(pv >= 0));
    if (np <= 0) break;  // unreachable: every level keeps >= 1 parent
    // t is the same in every lane: so are the level's sizes (scalar loops)
    const int ct = uniform((int)((t / P.pw) & (CR - 1)));
    const int nc = ((np - 1) << crlg) + ct + 1;
    const int apos = nc - 1;
    const int nt = wide ? (nc + 15) >> 4 : np;
    if (a.parents && lane < TK)
      a.parents[((((int64_t)l * a.B + b) * a.T + t) * a.Hkv + h) * TK + lane] = pv;
    if (SEL && l == 0) break;  // the bottom level selects nothing
    const int64_t hrow = ((int64_t)b * a.Hkv + h) * P.Np;
    const uint16_t* KH = P.kh + hrow * D;
    const uint16_t* KL = P.kl + hrow * D;
    const uint16_t* VH = P.vh + hrow * D;
    const uint16_t* VL = PREC ? P.vl + hrow * D : nullptr;
    const int32_t* pc = W.par[cur];
    auto node0_of = [&](int tau) {  // (the list is in pv: lane s holds parent s)
      const int s = wide ? (tau << 4) >> crlg : tau;
      return (__builtin_amdgcn_readlane(pv, s) << crlg) + (wide ? ((tau << 4) & (CR - 1)) : 0);
    };
    auto kload = [&](int tau, bf16x8 (&kh)[KS], bf16x8 (&kl)[KS]) {
      const int posk = wide ? (tau << 4) + u16 : (tau << crlg) + u16;
      const bool cvk = u16 < CRU && posk < nc;
      const int node0 = node0_of(tau), c = cvk ? u16 : 0;
      load_kfrag<D>(KH, node0, c, kg, kh);
      load_kfrag<D>(KL, node0, c, kg, kl);
    };

    // ---- scores of every tile (descending slot), S^T into LDS
    float qr[KS][8];
    qin.get(qr, a.scale);
    rot_by<D>(qr, a.cosb + (int64_t)ct * HALF, a.sinb + (int64_t)ct * HALF, kg);
    int cur_slot = uniform(wide ? ((nt - 1) << 4) >> crlg : nt - 1);
    float lmax = -INFINITY;
    auto score = [&](int tau, const bf16x8 (&kh)[KS], const bf16x8 (&kl)[KS]) {
      const int s = uniform(wide ? (tau << 4) >> crlg : tau);
      if (s != cur_slot) {
        rot_by<D>(qr, rot_cr[0], rot_cr[1], kg);
        cur_slot = s;
      }
      bf16x8 qh[KS], ql[KS];
      to_bf_split<D>(qr, qh, ql);
      f32x4 S = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int m = 0; m < KS; ++m) {
        S = mma32(kh[m], qh[m], S);
        S = mma32(kl[m], qh[m], S);
        S = mma32(kh[m], ql[m], S);
      }
      if (!wide || tau == nt - 1) {  // the other tiles hold 16 candidates
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int cu = 4 * kg + r;
          const int pos = wide ? (tau << 4) + cu : (tau << crlg) + cu;
          S[r] = cu < CRU && pos < nc ? S[r] : -INFINITY;
        }
      }
      lmax = fmaxf(lmax, fmaxf(fmaxf(S[0], S[1]), fmaxf(S[2], S[3])));
      W.st[tau][lane] = S;
    };
    for (int tau = nt - 1; tau >= 0; --tau) {
      bf16x8 kh[KS], kl[KS];
      kload(tau, kh, kl);
      score(tau, kh, kl);
    }

    if (l > 0) {
      // ---- importance sum_g exp(s - M), M = max over the level's scores
      const float M = wave_max_uniform(lmax);
      for (int tau = 0; tau < nt; ++tau) {
        const f32x4 S = W.st[tau][lane];
        float x[4], e[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          x[r] = (S[r] - M) * kLog2e;
          e[r] = __builtin_amdgcn_exp2f(x[r]);
        }
        // subnormal results (exp_sel), one wave test for the tile
        if (__builtin_expect(__any(fminf(fminf(x[0], x[1]), fminf(x[2], x[3])) < -126.f), 0)) {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (x[r] < -126.f) e[r] = __builtin_amdgcn_exp2f(x[r] + 64.f) * 5.42101086242752217e-20f;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) e[r] *= hv;
        // sum over the row's 16 lanes (heads) of each candidate r, by
        // recursive halving: lane bit 0 keeps r in {0,1} or {2,3}, bit 1 one
        // of those, then the four quads add up; lane u16 ends with candidate
        // r = 2 (u16 & 1) + ((u16 >> 1) & 1)
        const bool b0 = u16 & 1, b1 = (u16 >> 1) & 1;
        const float k0 = b0 ? e[2] : e[0], k1 = b0 ? e[3] : e[1];
        const float s0 = b0 ? e[0] : e[2], s1 = b0 ? e[1] : e[3];
        const float h0 = k0 + dpp<0xB1>(s0), h1 = k1 + dpp<0xB1>(s1);
        float c = (b1 ? h1 : h0) + dpp<0x4E>(b1 ? h0 : h1);
        c += dpp<0x124>(c);   // row rotate right by 4
        c += dpp<0x128>(c);   // row rotate right by 8
        if (u16 < 4) W.imp[(tau << 4) + 4 * kg + 2 * b0 + b1] = c;
      }
      if (pair) {
        // the pair's importance: both halves' sums taken to the pair's max
        // (the group-shared sum of src/naive.py:204-205 over all G heads)
        if (lane == 0) W.lvl_max = M;
        __syncthreads();
        const WaveLdsR& W0 = lds_all[wv & ~1];
        const WaveLdsR& W1 = lds_all[wv | 1];
        const float m0 = W0.lvl_max, m1 = W1.lvl_max, mp = fmaxf(m0, m1);
        select_topk<4>(W0.imp, nt, nc, apos, TK, wide, crlg, CR, CRU, W.par[cur],
                       W.par[cur ^ 1], W.selmask, lane, W1.imp, expf(m0 - mp), expf(m1 - mp));
        __syncthreads();  // the partner has read this wave's importances
      } else {
        wave_sync();
        select_topk<4>(W.imp, nt, nc, apos, TK, wide, crlg, CR, CRU, W.par[cur],
                       W.par[cur ^ 1], W.selmask, lane);
        wave_sync();
      }
    }
    if constexpr (SEL) {
      cur ^= 1;
      continue;
    }

    // ---- per-head max over the accumulated candidates (rows kg via LDS)
    const bool upper = l > 0;
    auto masked = [&](int tau) {
      f32x4 S = W.st[tau][lane];
      if (upper) {
        const int w = uniform((int)(W.selmask[tau >> 2] >> (16 * (tau & 3))));
#pragma unroll
        for (int r = 0; r < 4; ++r) {  // -inf where the candidate is passed down
          const uint32_t m = (uint32_t)__builtin_amdgcn_sbfe(w, 4 * kg + r, 1);
          S[r] = __uint_as_float((m & 0xff800000u) | (~m & __float_as_uint(S[r])));
        }
      }
      return S;
    };
    float gmx = lmax;  // the bottom level accumulates every candidate: the scores' max
    if (upper) {
      gmx = -INFINITY;
      for (int tau = 0; tau < nt; ++tau) {
        const f32x4 S = masked(tau);
        gmx = fmaxf(fmaxf(gmx, fmaxf(S[0], S[1])), fmaxf(S[2], S[3]));
      }
    }
    gmx = max_xor32(max_xor16(gmx));  // over the lane groups (candidates) of the head
    if (TRACE) {
      m_run = -INFINITY;
      l_part = 0.f;
#pragma unroll
      for (int n = 0; n < ND; ++n) O[n] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const float mnew = fmaxf(m_run, gmx);
    const float mref = mnew == -INFINITY ? 0.f : mnew;
    if (a.scores) {
      // every tile's scores relative to the head's running max, for the
      // backward (the accumulated ones are <= 0 there; fp16 RNE)
      const int64_t lg = (int64_t)l * a.B * a.T * a.Hkv + ((int64_t)b * a.T + t) * a.Hkv + h;
      // tile layout S[head][cand] (fp16, 16 x 16): this lane's candidates
      // 4kg..4kg+3 of head u16
      uint16_t* so = a.scores + lg * a.max_tiles * 256 + u16 * 16 + kg * 4;
      for (int tau = 0; tau < nt; ++tau) {
        const f32x4 S = W.st[tau][lane];
        uint32_t hb[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) hb[r] = __builtin_bit_cast(uint16_t, (_Float16)(S[r] - mref));
        *(uint2*)(so + tau * 256) = make_uint2(hb[0] | (hb[1] << 16), hb[2] | (hb[3] << 16));
      }
      if (kg == 0) a.smref[lg * 16 + u16] = mref;
    }
    const float alpha = __builtin_amdgcn_exp2f((m_run - mref) * kLog2e);
    m_run = mnew;
    l_part *= alpha;
#pragma unroll
    for (int n = 0; n < ND; ++n) O[n] *= alpha;

    // ---- O^T += V^T P^T over the tiles, V double-buffered
    auto vload = [&](int tau, s16x4 (&vh)[ND], s16x4 (&vl)[ND]) {
      const int vn = node0_of(tau) + (4 * kg < CRU ? 4 * kg : 0);
      // dims 32j + 2 u16 and 32j + 2 u16 + 1 (tiles 2j, 2j + 1): 16 bytes
      const int64_t vbase = (int64_t)(vn >> 4) * 16 * D + ((vn & 15) >> 2) * 4 * D + u16 * 8;
#pragma unroll
      for (int j = 0; j < ND / 2; ++j) {
        const uint4 w = *(const uint4*)(VH + vbase + (int64_t)j * 128);
        vh[2 * j] = __builtin_bit_cast(s16x4, make_uint2(w.x, w.y));
        vh[2 * j + 1] = __builtin_bit_cast(s16x4, make_uint2(w.z, w.w));
        if (PREC) {
          const uint4 wl = *(const uint4*)(VL + vbase + (int64_t)j * 128);
          vl[2 * j] = __builtin_bit_cast(s16x4, make_uint2(wl.x, wl.y));
          vl[2 * j + 1] = __builtin_bit_cast(s16x4, make_uint2(wl.z, wl.w));
        }
      }
    };
    auto pv_tile = [&](int tau, const s16x4 (&vh)[ND], const s16x4 (&vl)[ND]) {
      const f32x4 S = masked(tau);
      float p[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) p[r] = __builtin_amdgcn_exp2f((S[r] - mref) * kLog2e);
      l_part += (p[0] + p[1]) + (p[2] + p[3]);
      s16x4 ph, pl;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const uint16_t hb = f_to_bf(p[r]);
        ph[r] = (short)hb;
        pl[r] = PREC ? f_to_bfs(p[r] - bf_to_f(hb)) : (short)0;
      }
#pragma unroll
      for (int n = 0; n < ND; ++n) {
        O[n] = mma16(vh[n], ph, O[n]);
        if (PREC) {
          O[n] = mma16(vh[n], pl, O[n]);
          O[n] = mma16(vl[n], ph, O[n]);
        }
      }
    };
    {
      s16x4 av[ND], avl[ND], bv[ND], bvl[ND];
      vload(0, av, avl);
      if (nt >= 2) vload(1, bv, bvl);
      for (int tau = 0; tau < nt; tau += 2) {
        pv_tile(tau, av, avl);
        if (tau + 2 < nt) vload(tau + 2, av, avl);
        if (tau + 1 < nt) {
          pv_tile(tau + 1, bv, bvl);
          if (tau + 3 < nt) vload(tau + 3, bv, bvl);
        }
      }
    }
    if (TRACE)
      trace_store<D>(a, l, ((int64_t)b * a.T + t) * a.H + h * G + u16, gv, kg, m_run, l_part, O);
    cur ^= 1;
  }

  if constexpr (SEL) return;
  float lt;
  if (TRACE) {
    lt = trace_merge<D>(a, ((int64_t)b * a.T + t) * a.H + h * G + u16, gv, kg, m_run, O);
  } else {
    lt = add_xor32(add_xor16(l_part));
  }
  if (gv) {
    const int64_t hq = ((int64_t)b * a.T + t) * a.H + h * G + u16;
    const float inv = 1.f / lt;
    store_out<D, TIn>((TIn*)a.out + hq * D, kg, O, [&](float x) { return x * inv; });
    if (kg == 0) {
      a.gmax[hq] = m_run;
      a.gsum[hq] = lt;
    }
  }
}

static void launch_fwd_reg(int D, int dtype, const FwdArgs& a, dim3 grid, hipStream_t st, bool sel) {
  for_dim_type(D, dtype, [&](auto d, auto prec, auto* tin) {
    using TIn = typename std::remove_pointer<decltype(tin)>::type;
    constexpr int DD = decltype(d)::value;
    constexpr bool PREC = decltype(prec)::value;
    if (sel)
      hipLaunchKernelGGL((fwd_reg_kernel<DD, PREC, TIn, false, true>), grid, dim3(256), 0, st, a);
    else if (a.tout != nullptr)
      hipLaunchKernelGGL((fwd_reg_kernel<DD, PREC, TIn, true>), grid, dim3(256), 0, st, a);
    else
      hipLaunchKernelGGL((fwd_reg_kernel<DD, PREC, TIn, false>), grid, dim3(256), 0, st, a);
  });
}

}  // namespace htree

using namespace htree;

static int forward_impl(const htree_dims* d, float scale, const void* q, const void* tree_ws,
                        int64_t tree_ws_bytes, const float* cos_table, const float* sin_table,
                        void* out, float* gmax, float* gsum, int32_t* parents, void* scores,
                        int64_t scores_bytes, float* tmax, float* tsum, float* tout,
                        void* stream, bool sel = false) {
  Plan P;
  int rc = make_plan(d, &P);
  if (rc) return rc;
  if (!q || !tree_ws || !cos_table || !sin_table) return HTREE_ENULL;
  // the selection-only launch writes the lists alone
  if (sel ? !parents : (!out || !gmax || !gsum)) return HTREE_ENULL;
  if (sel) scores = nullptr, tout = nullptr;
  if (tree_ws_bytes < P.bytes) return HTREE_EWORKSPACE;
  if (P.split)  // the shared selection does not fit one block
    return split_forward(d, P, scale, q, tree_ws, cos_table, sin_table, out, gmax, gsum, parents,
                         tmax, tsum, tout, stream, sel);
  int64_t off_mref = 0;
  const int64_t sbytes = train_scores_bytes(d, P, &off_mref);
  if (scores && sbytes == 0) scores = nullptr;  // this configuration recomputes in the backward
  if (scores && scores_bytes < sbytes) return HTREE_EWORKSPACE;
  const bool wide_fwd = P.wide || d->kv_share == 4;  // one block per kv_share KV heads
  FwdArgs a;
  memset(&a, 0, sizeof(a));
  const char* base = (const char*)tree_ws;
  for (int l = 0; l < P.L; ++l) {
    // the wide forward accumulates from KH / KL (the top level's at the angle
    // of the node) and selects from SH / SL, which a level that selects
    // nothing may lack; for the other forms the two are one
    a.lv[l].kh = (const uint16_t*)(base + (P.off_kh[l]));
    a.lv[l].kl = (const uint16_t*)(base + (P.off_kl[l]));
    a.lv[l].sh = P.off_sh[l] >= 0 ? (const uint16_t*)(base + P.off_sh[l]) : nullptr;
    a.lv[l].sl = P.off_sl[l] >= 0 ? (const uint16_t*)(base + P.off_sl[l]) : nullptr;
    a.lv[l].vh = (const uint16_t*)(base + P.off_vh[l]);
    a.lv[l].vl = P.off_vl[l] >= 0 ? (const uint16_t*)(base + P.off_vl[l]) : nullptr;
    a.lv[l].N = P.N[l];
    a.lv[l].Np = P.Np[l];
    a.lv[l].pw = P.pw[l];
  }
  a.q = q;
  a.out = out;
  a.gmax = gmax;
  a.gsum = gsum;
  a.parents = parents;
  a.scores = (uint16_t*)scores;
  a.smref = scores ? (float*)((char*)scores + off_mref) : nullptr;
  a.tmax = tmax;
  a.tsum = tsum;
  a.tout = tout;
  a.max_tiles = P.max_tiles;
  a.cosb = cos_table;
  a.sinb = sin_table;
  a.B = d->B;
  a.T = d->T;
  a.H = d->H;
  a.Hkv = d->H_kv;
  a.G = d->H / d->H_kv;
  a.CR = d->compression_rate;
  a.crlg = P.cr_log2;
  a.TK = d->top_k;
  a.L = P.L;
  a.scale = scale;
  a.kv_share = d->kv_share > 1 ? d->kv_share : 1;
  a.gpad = d->group_pad;
  // the streaming kernel addresses one (b, h_kv) block of a level array
  // with 32-bit byte offsets
  if (!wide_fwd && (P.max_tiles > 16 || a.gpad > 0) && P.Np[0] * d->D * 2 > 0x7fffffffll)
    return HTREE_EUNSUPPORTED;
  const int64_t groups = (int64_t)d->B * d->H_kv * d->T;
  // blocks dealt round-robin to the 8 XCDs: XCD x gets blocks x, x+8, ...,
  // which map to a contiguous range of query groups (one tree per XCD's L2)
  const int64_t nblk = wide_fwd ? groups / a.kv_share
                                : (groups + kWavesPerBlock - 1) / kWavesPerBlock;
  const int64_t per = (nblk + 7) / 8;
  if (per * 8 > 0x7fffffff) return HTREE_EUNSUPPORTED;
  a.per_xcd = (int32_t)per;
  const dim3 grid((unsigned)(per * 8));
  hipStream_t st = (hipStream_t)stream;
  if (wide_fwd)
    d->D == 256 ? launch_fwd_wide_d<256>(d->dtype, a, grid, st, sel)
    : d->D == 128 ? launch_fwd_wide_d<128>(d->dtype, a, grid, st, sel)
    : d->D == 32 ? launch_fwd_wide_d<32>(d->dtype, a, grid, st, sel)
                 : launch_fwd_wide_d<64>(d->dtype, a, grid, st, sel);
  else if (P.max_tiles <= 16 && a.gpad == 0)  // (padding heads: the streaming form)
    launch_fwd_reg(d->D, d->dtype, a, grid, st, sel);
  else
    launch_fwd_stream(d->D, d->dtype, a, grid, st, sel);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? HTREE_OK : (int)e;
}

extern "C" int htree_forward(const htree_dims* d, float scale, const void* q,
                             const void* tree_ws, int64_t tree_ws_bytes,
                             const float* cos_table, const float* sin_table, void* out,
                             float* gmax, float* gsum, int32_t* parents, void* stream) {
  return forward_impl(d, scale, q, tree_ws, tree_ws_bytes, cos_table, sin_table, out, gmax, gsum,
                      parents, nullptr, 0, nullptr, nullptr, nullptr, stream);
}

extern "C" int htree_train_scores_bytes(const htree_dims* d, int64_t* bytes) {
  Plan P;
  int rc = make_plan(d, &P);
  if (rc) return rc;
  if (!bytes) return HTREE_ENULL;
  *bytes = train_scores_bytes(d, P, nullptr);
  return HTREE_OK;
}

extern "C" int htree_forward_train(const htree_dims* d, float scale, const void* q,
                                   const void* tree_ws, int64_t tree_ws_bytes,
                                   const float* cos_table, const float* sin_table, void* out,
                                   float* gmax, float* gsum, int32_t* parents, void* scores,
                                   int64_t scores_bytes, void* stream) {
  if (!parents) return HTREE_ENULL;
  return forward_impl(d, scale, q, tree_ws, tree_ws_bytes, cos_table, sin_table, out, gmax, gsum,
                      parents, scores, scores_bytes, nullptr, nullptr, nullptr, stream);
}

extern "C" int htree_forward_trace(const htree_dims* d, float scale, const void* q,
                                   const void* tree_ws, int64_t tree_ws_bytes,
                                   const float* cos_table, const float* sin_table, void* out,
                                   float* gmax, float* gsum, int32_t* parents, float* level_max,
                                   float* level_sum, float* level_out, void* stream) {
  if (!parents || !level_max || !level_sum || !level_out) return HTREE_ENULL;
  return forward_impl(d, scale, q, tree_ws, tree_ws_bytes, cos_table, sin_table, out, gmax, gsum,
                      parents, nullptr, 0, level_max, level_sum, level_out, stream);
}

extern "C" int htree_select(const htree_dims* d, float scale, const void* q, const void* tree_ws,
                            int64_t tree_ws_bytes, const float* cos_table, const float* sin_table,
                            int32_t* parents, void* stream) {
  return forward_impl(d, scale, q, tree_ws, tree_ws_bytes, cos_table, sin_table, nullptr, nullptr,
                      nullptr, parents, nullptr, 0, nullptr, nullptr, nullptr, stream, true);
}
