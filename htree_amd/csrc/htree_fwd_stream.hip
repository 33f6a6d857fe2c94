// Streaming form of the fused forward (htree_fwd.hip describes the work the
// fused forwards share).
#include "htree_fwd.h"

namespace htree {

template <int MAXSLOT>
struct WaveLds {
  int32_t par[2][kMaxTK];
  float imp[MAXSLOT * 64];
  float mt[MAXSLOT * 4];
  unsigned long long selmask[MAXSLOT];
  float lvl_max;  // the level's final running max (KV-head pairs)
};

// One tile's inputs staged in LDS: the 16-node K~ blocks (hi, lo) and the
// V^T block (hi, lo) that hold the tile, as they lie in the packed tree (an
// operand read's 64 lanes take 1 KB in a row: no bank conflicts).
template <int D, bool PREC>
struct FwdStage {
  static constexpr int KB = 16 * D * 2;           // K~ block of 16 nodes (bf16)
  static constexpr int OFF_KL = KB;
  static constexpr int VB = 16 * D * 2;           // V^T block of 16 nodes (bf16)
  static constexpr int OFF_V = 2 * KB;
  static constexpr int OFF_VL = OFF_V + VB;
  static constexpr int BYTES = OFF_V + (PREC ? 2 : 1) * VB;
};

// Copies of one tile's inputs into a wave's LDS slot (FwdStage layout) by
// buffer loads over one (b, h_kv) block of the level arrays: offsets past
// the block read as zero, so rows past the level's nodes are harmless (their
// scores are masked).  The lane offsets are recomputed per call (an opaque
// copy of the lane index) instead of being hoisted and held in registers.
template <int D, bool PREC>
struct TileStage {
  using St = FwdStage<D, PREC>;
  char* slot;
  __amdgpu_buffer_rsrc_t rkh, rkl, rvh, rvl;

  __device__ __forceinline__ void issue(int node0, bool with_v, int lane) const {
    int ln = lane;
    asm volatile("" : "+v"(ln));
    const int koff = (node0 >> 4) * St::KB;
#pragma unroll
    for (int j = 0; j < St::KB / 1024; ++j) {
      const int off = koff + (j * 64 + ln) * 16;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rkh, (lds_void*)(slot + j * 1024), 16, off, 0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rkl, (lds_void*)(slot + St::OFF_KL + j * 1024), 16,
                                               off, 0, 0, 0);
    }
    if (with_v) {
      const int voff = (node0 >> 4) * St::VB;
#pragma unroll
      for (int j = 0; j < St::VB / 1024; ++j) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rvh, (lds_void*)(slot + St::OFF_V + j * 1024), 16,
                                                 voff + (j * 64 + ln) * 16, 0, 0, 0);
        if (PREC)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rvl, (lds_void*)(slot + St::OFF_VL + j * 1024), 16,
                                                   voff + (j * 64 + ln) * 16, 0, 0, 0);
      }
    }
  }
  static __device__ __forceinline__ void wait_copies() {
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the slot's copies have landed
    __builtin_amdgcn_wave_barrier();
  }
  static __device__ __forceinline__ void reads_done() {
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the slot's reads have completed
    __builtin_amdgcn_wave_barrier();
  }
  // K~ fragments of node c of the staged block, the lane group's d-slots
  __device__ __forceinline__ void kread(bf16x8 (&kh)[D / 32], bf16x8 (&kl)[D / 32], int c,
                                        int lane) const {
    int ln = lane;
    asm volatile("" : "+v"(ln));
    const char* row = slot + c * 16 + (ln >> 4) * 256;
#pragma unroll
    for (int m = 0; m < D / 32; ++m) {
      kh[m] = *(const bf16x8*)(row + m * 1024);
      kl[m] = *(const bf16x8*)(row + St::OFF_KL + m * 1024);
    }
  }
  // V^T fragments: nodes c0 .. c0+3 (one quad, c0 % 4 == 0) of the staged
  // block, output tiles 2j and 2j + 1 at dims 32j + 2 u16 and 32j + 2 u16 + 1
  // (odim) in one 16-byte read: the 16 lanes of a lane group read 256
  // contiguous bytes (no bank conflicts)
  __device__ __forceinline__ void vread(s16x4 (&vh)[D / 16], s16x4 (&vl)[D / 16], int c0,
                                        int u16) const {
#pragma unroll
    for (int j = 0; j < D / 32; ++j) {
      const int e = (c0 >> 2) * 4 * D + (32 * j + 2 * u16) * 4;
      const uint4 w = *(const uint4*)(slot + St::OFF_V + e * 2);
      vh[2 * j] = __builtin_bit_cast(s16x4, make_uint2(w.x, w.y));
      vh[2 * j + 1] = __builtin_bit_cast(s16x4, make_uint2(w.z, w.w));
      if (PREC) {
        const uint4 wl = *(const uint4*)(slot + St::OFF_VL + e * 2);
        vl[2 * j] = __builtin_bit_cast(s16x4, make_uint2(wl.x, wl.y));
        vl[2 * j + 1] = __builtin_bit_cast(s16x4, make_uint2(wl.z, wl.w));
      }
    }
  }
};

// Streaming forward for levels of 17..64 candidate tiles (e.g. top_k 32 with
// CR 32): one wave per query group; upper levels score every tile for the
// importance, select, then score again for the accumulation.  Each tile's
// K~ rows (and, for the accumulation, its V^T block) are copied into the
// wave's LDS slot by buffer loads (range-checked against the level's
// (b, h_kv) rows) one tile ahead: the copies of tile tau+1 are issued as
// soon as tile tau's fragments have moved to registers, and land while tile
// tau is computed.  Tiles run in ascending parent slot and the query turns
// by R(., -CR) per slot (a table row in LDS), so a tile reads no global
// memory besides its copies.
// Bound by its vector ALU work per tile (T 131072, 64/8 heads, D 128, CR 32):
// the turned query is split once per slot instead of once per tile, the
// subnormal test is one per tile, a tile's masks are formed only at a level's
// last tile, the passed-down candidates start their scores at -inf, and the
// rescale runs only where a head's max rises: 132.1 -> 124.4 ms; 126 ms with
// the scores in their own units, in which gmax is a score and the backward's P
// sums to one (with log2 e in the query fp32 gradients of clustered keys were
// 18 to 25% further from float64).
template <int D, bool PREC, typename TIn, int MAXSLOT, bool TRACE, bool SEL = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D == 256 ? 1 : 2))) void fwd_kernel(const FwdArgs a) {
  static_assert(!(SEL && TRACE), "selection only: no trace");
  constexpr int KS = D / 32, ND = D / 16, HALF = D / 2;
  using St = FwdStage<D, PREC>;
  __shared__ WaveLds<MAXSLOT> lds_all[kWavesPerBlock];
  __shared__ __attribute__((aligned(16))) char stage_all[kWavesPerBlock][St::BYTES];
  __shared__ float rot_m[2][HALF];  // cos(CR theta), -sin(CR theta)

  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int u16 = lane & 15, kg = lane >> 4;
  const int G = a.G, CR = a.CR, crlg = a.crlg, TK = a.TK;
  if (threadIdx.x < HALF) {
    rot_m[0][threadIdx.x] = a.cosb[(int64_t)CR * HALF + threadIdx.x];
    rot_m[1][threadIdx.x] = -a.sinb[(int64_t)CR * HALF + threadIdx.x];
  }
  __syncthreads();
  // XCD-aware order: hardware deals blocks round-robin over the 8 XCDs; give
  // each XCD a contiguous range of query groups (same (b, h_kv) tree).
  const int bid = blockIdx.x;
  const int64_t lb = (int64_t)(bid & 7) * a.per_xcd + (bid >> 3);
  const int64_t grp = lb * kWavesPerBlock + wv;
  // KV-head pairs (kv_share 2): as in fwd_reg_kernel, waves 2i and 2i+1 take
  // KV heads 2h, 2h+1 of one query and meet at two block barriers per upper
  // level; the waves of an empty pair pass the same barriers
  const bool pair = a.kv_share == 2;
  if (grp >= (int64_t)a.B * a.Hkv * a.T) {
    if (pair)
      for (int l = a.L - 1; l >= 1; --l) {
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
  const int Gs = sel_heads(a, h);  // heads in the selection
  WaveLds<MAXSLOT>& W = lds_all[wv];
  char* slot = stage_all[wv];
  const int CRU = CR < 16 ? CR : 16;
  const bool wide = CR >= 16;

  // Query rows past the group repeat its heads: their scores stay in the
  // range of the others, and they are left out of the sums and not stored.  (A
  // padded group's are zero and masked, as its padding heads.)
  const bool gv = u16 < G;
  const TIn* qp = (const TIn*)a.q +
                  (((int64_t)b * a.T + t) * a.H + h * G + (gv ? u16 : a.gpad > 0 ? 0 : u16 % G)) * D;

  float m_run = -INFINITY, l_part = 0.f;
  f32x4 O[ND];
#pragma unroll
  for (int n = 0; n < ND; ++n) O[n] = f32x4{0.f, 0.f, 0.f, 0.f};

  // virtual parents of the top level (src/naive.py:108-118)
  {
    const int64_t nvp = (t / a.lv[a.L - 1].pw) / CR + 1;
    if (lane < TK) W.par[0][lane] = lane < nvp ? lane : -1;
  }
  int cur = 0;

  for (int l = a.L - 1; l >= 0; --l) {
    wave_sync();
    const LevelPtrs P = a.lv[l];
    const int pv = lane < TK ? W.par[cur][lane] : -1;
    const int np = __popcll(__ballot(pv >= 0));
    if (np <= 0) break;  // unreachable: every level keeps >= 1 parent
    const int ct = (int)((t / P.pw) & (CR - 1));
    const int nc = ((np - 1) << crlg) + ct + 1;
    const int apos = nc - 1;
    const int nt = wide ? (nc + 15) >> 4 : np;
    if (a.parents && lane < TK)
      a.parents[((((int64_t)l * a.B + b) * a.T + t) * a.Hkv + h) * TK + lane] = pv;
    if (SEL && l == 0) break;  // the bottom level selects nothing
    const int64_t hrow = ((int64_t)b * a.Hkv + h) * P.Np;
    const int lvl_bytes = (int)(P.Np * D * 2);  // one (b, h_kv) block of a level array
    const TileStage<D, PREC> stg{slot, buf_rsrc(P.kh + hrow * D, lvl_bytes),
                                 buf_rsrc(P.kl + hrow * D, lvl_bytes),
                                 buf_rsrc(P.vh + hrow * D, lvl_bytes),
                                 buf_rsrc((PREC ? P.vl : P.vh) + hrow * D, lvl_bytes)};
    const bool upper = l > 0;
    auto slot_of = [&](int tau) { return wide ? (tau << 4) >> crlg : tau; };
    auto node0_of = [&](int tau) {
      return (W.par[cur][slot_of(tau)] << crlg) + (wide ? ((tau << 4) & (CR - 1)) : 0);
    };
    auto issue = [&](int tau, bool with_v) { stg.issue(node0_of(tau), with_v, lane); };
    auto wait_copies = [&]() { stg.wait_copies(); };
    auto reads_done = [&]() { stg.reads_done(); };
    // node of the staged block: the tile's candidate u16 (CR < 16: the
    // tile starts inside the block)
    auto kread = [&](int tau, bf16x8 (&kh)[KS], bf16x8 (&kl)[KS]) {
      const int c = wide ? u16 : (node0_of(tau) & 15) + (u16 < CRU ? u16 : 0);
      stg.kread(kh, kl, c, lane);
    };
    // the query turned to a slot, R(q, apos) at slot 0, -CR per slot after,
    // and split once per slot (a slot has CR / 16 tiles; at D = 256 once per
    // tile, as the registers do not hold both)
    constexpr bool ONCE = D <= 128;
    float qr[KS][8];
    bf16x8 qh[KS], ql[KS];
    int cur_slot = 0;
    auto frame_start = [&](const TIn* p, bool live) {
      // (read again at each pass: held, its registers spill at D = 128)
      QFrag<D, TIn, false> qin;
      qin.load(p, kg, live);
      qin.get(qr, a.scale);
      rot_by<D>(qr, a.cosb + (int64_t)apos * HALF, a.sinb + (int64_t)apos * HALF, kg);
      if (ONCE) to_bf_split<D>(qr, qh, ql);
      cur_slot = 0;
    };
    auto frame_to = [&](int s) {
      if (cur_slot < s) {  // (tiles are taken in order: one slot on)
        rot_by<D>(qr, rot_m[0], rot_m[1], kg);
        if (ONCE) to_bf_split<D>(qr, qh, ql);
        cur_slot = s;
      }
      if (!ONCE) to_bf_split<D>(qr, qh, ql);
    };

    // ------------------------------------------------ selection (upper levels)
    if (upper) {
      float Mrun = -INFINITY;
      float hm[4];  // 1 for heads 4kg + r of the selection (formed per level)
      {
        int kq = kg;
        asm volatile("" : "+v"(kq));
#pragma unroll
        for (int r = 0; r < 4; ++r) hm[r] = 4 * kq + r < Gs ? 1.f : 0.f;
      }
      // (rows past the heads of the selection repeat them here: no row's
      // score is out of the range of the others)
      frame_start(a.gpad == 0 ? qp : qp + (u16 < Gs ? 0 : u16 % Gs - (gv ? u16 : 0)) * D, true);
      issue(0, false);
      for (int tau = 0; tau < nt; ++tau) {
        frame_to(slot_of(tau));
        wait_copies();
        bf16x8 kh[KS], kl[KS];
        kread(tau, kh, kl);
        reads_done();
        if (tau + 1 < nt) issue(tau + 1, false);
        f32x4 S = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int m = 0; m < KS; ++m) {
          S = mma32(qh[m], kh[m], S);
          S = mma32(qh[m], kl[m], S);
          S = mma32(ql[m], kh[m], S);
        }
        // S[r] = score[g = 4kg + r][candidate u16].  A column that is no
        // candidate is kept out of the max and its sum not read; its scores
        // (of some node of the tree) stay as they are, so that the subnormal
        // test below sees no -inf
        float tm = fmaxf(fmaxf(S[0], S[1]), fmaxf(S[2], S[3]));
        if (!wide || tau == nt - 1) {
          const int pos = wide ? (tau << 4) + u16 : (tau << crlg) + u16;
          tm = u16 < CRU && pos < nc ? tm : -INFINITY;
        }
        Mrun = fmaxf(Mrun, wave_max(tm));
#pragma unroll
        for (int r = 0; r < 4; ++r) S[r] = (S[r] - Mrun) * kLog2e;
        // subnormal results (exp_sel), one wave test for the tile
        if (__builtin_expect(__any(fminf(fminf(S[0], S[1]), fminf(S[2], S[3])) < -126.f), 0)) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const bool sb = S[r] < -126.f;
            const float p = __builtin_amdgcn_exp2f(sb ? S[r] + 64.f : S[r]);
            S[r] = sb ? p * 5.42101086242752217e-20f : p;
          }
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) S[r] = __builtin_amdgcn_exp2f(S[r]);
        }
        float e = 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r) e = fmaf(S[r], hm[r], e);
        e = add_xor32(add_xor16(e));
        if (kg == 0) W.imp[(tau << 4) + u16] = e;
        if (lane == 0) W.mt[tau] = Mrun;
      }
      // a pair's importance: both halves' sums, each from its tile's running
      // max, taken to the pair's max (the group-shared sum of
      // src/naive.py:204-205 over all G heads), in a fixed order
      const WaveLds<MAXSLOT>& W0 = lds_all[wv & ~1];
      const WaveLds<MAXSLOT>& W1 = lds_all[wv | 1];
      float Mp = Mrun;
      if (pair) {
        if (lane == 0) W.lvl_max = Mrun;
        __syncthreads();
        Mp = fmaxf(W0.lvl_max, W1.lvl_max);
      } else {
        wave_sync();
      }

      // importance of position j lives in lane j % 64 of slot j / 64; the
      // key is the float's bit pattern + 1 (0 = no candidate), so unsigned
      // order is importance order and exact ties are resolved by position.
      const int take = TK < nc ? TK : nc;
      // lane-dependent offsets are recomputed per level rather than hoisted
      // out of the level loop and held (or spilled) across it
      int ln = lane;
      asm volatile("" : "+v"(ln));
      const int su = ln & 15, skg = ln >> 4;
      const int nslot = (nt + 3) >> 2;
      uint32_t key[MAXSLOT];
#pragma unroll
      for (int sl = 0; sl < MAXSLOT; ++sl) {
        key[sl] = 0u;
        if (sl < nslot) {
          const int tau = 4 * sl + skg;
          const int pos = wide ? (tau << 4) + su : (tau << crlg) + su;
          if (tau < nt && su < CRU && pos < nc) {
            float v;
            if (pos == apos) {
              v = 1e6f;  // rightmost candidate always kept (src/naive.py:93)
            } else if (pair) {
              v = W0.imp[64 * sl + ln] * expf(W0.mt[tau] - Mp) +
                  W1.imp[64 * sl + ln] * expf(W1.mt[tau] - Mp);
            } else {
              v = W.imp[64 * sl + ln];
              const float mt = W.mt[tau];
              if (mt != Mrun) v *= expf(mt - Mrun);
            }
            key[sl] = __float_as_uint(v) + 1u;
          }
        }
      }
      if (pair) __syncthreads();  // the partner has read this wave's importances
      uint32_t thr = 0u;
      for (int bit = 30; bit >= 0; --bit) {
        const uint32_t c = thr | (1u << bit);
        int cnt = 0;
#pragma unroll
        for (int sl = 0; sl < MAXSLOT; ++sl)
          if (sl < nslot) cnt += __popcll(__ballot(key[sl] >= c));
        if (cnt >= take) thr = c;
      }
      int ngt = 0;
#pragma unroll
      for (int sl = 0; sl < MAXSLOT; ++sl)
        if (sl < nslot) ngt += __popcll(__ballot(key[sl] > thr));
      const int need = take - ngt;
      int eq_before = 0, sel_before = 0;
      const int nxt = cur ^ 1;
#pragma unroll
      for (int sl = 0; sl < MAXSLOT; ++sl) {
        if (sl < nslot) {
          const unsigned long long em = __ballot(key[sl] == thr);
          const bool sel = key[sl] > thr || (key[sl] == thr && eq_before + mbcnt64(em) < need);
          const unsigned long long sm = __ballot(sel);
          if (lane == 0) W.selmask[sl] = sm;
          if (sel) {
            const int tau = 4 * sl + skg;
            const int s = wide ? (tau << 4) >> crlg : tau;
            const int node =
                (W.par[cur][s] << crlg) + (wide ? ((tau << 4) & (CR - 1)) : 0) + su;
            W.par[nxt][sel_before + mbcnt64(sm)] = node;
          }
          eq_before += __popcll(em);
          sel_before += __popcll(sm);
        }
      }
      if (lane >= take && lane < TK) W.par[nxt][lane] = -1;
      wave_sync();
    }
    if constexpr (SEL) {  // (the scoring pass left no copy in flight)
      cur ^= 1;
      continue;
    }

    // ------------------------------------------------ accumulation
    if (TRACE) {
      m_run = -INFINITY;
      l_part = 0.f;
#pragma unroll
      for (int n = 0; n < ND; ++n) O[n] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    frame_start(qp, gv || a.gpad == 0);
    issue(0, true);
    for (int tau = 0; tau < nt; ++tau) {
      frame_to(slot_of(tau));
      const int node0 = node0_of(tau);
      // -inf where the candidate is passed down
      f32x4 S = {0.f, 0.f, 0.f, 0.f};
      if (upper) {
        const int w = uniform((int)(W.selmask[tau >> 2] >> (16 * (tau & 3))));
#pragma unroll
        for (int r = 0; r < 4; ++r)
          S[r] = __int_as_float(__builtin_amdgcn_sbfe(w, 4 * kg + r, 1) & 0xff800000);
      }
      wait_copies();
      bf16x8 kh[KS], kl[KS];
      kread(tau, kh, kl);
      // V^T fragment: nodes node0 + 4kg + 0..3 of the staged block at d = 16n + u16
      const int c0 = (node0 & 15) + (4 * kg < CRU ? 4 * kg : 0);
      s16x4 vh[ND], vl[ND];
      stg.vread(vh, vl, c0, u16);
      reads_done();
      if (tau + 1 < nt) issue(tau + 1, true);
#pragma unroll
      for (int m = 0; m < KS; ++m) {
        S = mma32(kh[m], qh[m], S);
        S = mma32(kl[m], qh[m], S);
        S = mma32(kh[m], ql[m], S);
      }
      // S[r] = score[candidate 4kg + r][g = u16]
      if (!wide || tau == nt - 1) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int cu = 4 * kg + r;
          const int pos = wide ? (tau << 4) + cu : (tau << crlg) + cu;
          S[r] = cu < CRU && pos < nc ? S[r] : -INFINITY;
        }
      }
      float tm = fmaxf(fmaxf(S[0], S[1]), fmaxf(S[2], S[3]));
      tm = max_xor32(max_xor16(tm));
      if (!__any(tm > -INFINITY)) continue;  // every candidate of the tile passed down
      float alpha = 1.f;
      if (__any(tm > m_run)) {  // some head's max rises: rescale
        const float mnew = fmaxf(m_run, tm);
        alpha = mnew == -INFINITY ? 1.f : __builtin_amdgcn_exp2f((m_run - mnew) * kLog2e);
        m_run = mnew;
#pragma unroll
        for (int n = 0; n < ND; ++n) O[n] *= alpha;
      }
      const float mref = m_run == -INFINITY ? 0.f : m_run;
      float p[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) p[r] = __builtin_amdgcn_exp2f((S[r] - mref) * kLog2e);
      l_part = l_part * alpha + ((p[0] + p[1]) + (p[2] + p[3]));
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
    }
    wait_copies();  // no copy into the slot is left in flight past the level
    if (TRACE)
      trace_store<D>(a, l, ((int64_t)b * a.T + t) * a.H + h * G + u16, u16 < G, kg,
                           m_run, l_part, O);
    cur ^= 1;
  }

  if constexpr (SEL) return;
  // final normalisation (src/parallel.py:321-363): out = o / s
  float lt;
  if (TRACE) {
    lt = trace_merge<D>(a, ((int64_t)b * a.T + t) * a.H + h * G + u16, u16 < G, kg, m_run, O);
  } else {
    lt = add_xor32(add_xor16(l_part));
  }
  if (u16 < G) {
    const int64_t hq = ((int64_t)b * a.T + t) * a.H + h * G + u16;
    store_out<D, TIn>((TIn*)a.out + hq * D, kg, O, [&](float x) { return x / lt; });
    if (kg == 0) {
      a.gmax[hq] = m_run;
      a.gsum[hq] = lt;
    }
  }
}

void launch_fwd_stream(int D, int dtype, const FwdArgs& a, dim3 grid, hipStream_t st, bool sel) {
  for_dim_type(D, dtype, [&](auto d, auto prec, auto* tin) {
    using TIn = typename std::remove_pointer<decltype(tin)>::type;
    constexpr int DD = decltype(d)::value;
    constexpr bool PREC = decltype(prec)::value;
    if (sel)
      hipLaunchKernelGGL((fwd_kernel<DD, PREC, TIn, 16, false, true>), grid, dim3(256), 0, st, a);
    else if (a.tout != nullptr)
      hipLaunchKernelGGL((fwd_kernel<DD, PREC, TIn, 16, true>), grid, dim3(256), 0, st, a);
    else
      hipLaunchKernelGGL((fwd_kernel<DD, PREC, TIn, 16, false>), grid, dim3(256), 0, st, a);
  });
}

}  // namespace htree
