// The per-wave half of the one-wave-per-SIMD forward (attn_fwd.hip: four
// waves of 64 queries sharing K/V tiles; attn_fwd_ks.hip: four waves of the
// same 64 queries, each with key tiles of its own): 64 queries' operands,
// accumulators and softmax state, and the slot schedule of one 64-key tile.
// The reasons for the layout and the schedule stand in attn_fwd.hip.
#pragma once

#include <type_traits>

#include "attn_fwd.h"
#include "tile_io.h"

namespace aa {

constexpr uint32_t kVOff = kTileElems * sizeof(bf16);  // V tile past the K tile of a stage

// Operand reads ahead of their MFMA: K operands (each feeds the two MFMAs of
// a pair of slots) are read kKPf pairs ahead, V^T operands kVPf pairs ahead
// into a queue one entry longer than that needs (a V^T operand stays
// allocated for one slot after its last MFMA).
constexpr int kKPf = 2, kKQ = kKPf + 1;
constexpr int kVPf = 2, kVQ = kVPf + 2;
constexpr int kread_slot(int j) { return j < kKPf ? 0 : 2 * (j - kKPf); }
constexpr int vread_slot(int pp) { return 32 + 2 * (pp - kVPf); }
// P unit u (2 scores of query block (u >> 2) & 1, key chunk u >> 3) starts in
// slot 3u / 2 and ends two slots later (slots 0-48); the P operand of chunk c4
// is first used in slot 32 + 8 c4, after its last unit. Max steps of the next
// tile: slots 48-63.
constexpr int exp_slot(int u) { return (3 * u) / 2; }
constexpr int kMaxSlot0 = 48;
// O^T += V^T P^T with O in AGPRs, as inline asm: the builtin would follow the
// function-wide choice of one register file for every MFMA accumulator, and S
// must stay in VGPRs for the softmax. O is only read or written by VALU code
// behind fence_o(), and the A/B operands are read when the MFMA issues.
__device__ __forceinline__ void mfma_pv(f32x16& acc, bf16x8 a, bf16x8 b) {
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}
__device__ __forceinline__ void keep_alive(bf16x8 v) { asm volatile("" ::"v"(v)); }
// Row sums (the accumulator and the 0/1 selector in AGPRs, as for O).
__device__ __forceinline__ void mfma_rowsum(f32x4& acc, bf16x8 sel, bf16x8 p) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "a"(sel), "v"(p));
}

// Per-wave state and work: 64 queries (blocks qb = 0, 1 of 32), their Q^T
// operands, O^T accumulators and running softmax statistics.
struct FwdWave {
  bf16x8 qreg[2][8];  // Q^T (qb, kk): lane holds Q[32 qb + li][16 kk + 8 hh + 0..7]; AGPRs
  f32x16 o[4][2];     // O^T (dt, qb): d = 32 dt + rows, query 32 qb + li; AGPRs
  f32x16 s[2][2][2];  // S^T (buffer, kb, qb): keys 32 kb + rows of the tile, query 32 qb + li
  bf16x8 pb[4][2];    // P^T (c4, qb): keys 16 c4 + .. of the tile, in accumulator order
  float m_raw[2];     // running max of query 32 qb + li, raw score units
  float mt[2];        // row max of the next tile (raw)
  f32x4 lsum[2];      // row sum of query 32 qb + li (all four elements), by MFMA
  float lf[2][2];     // with FSUM: this lane's sums of the fp32 probabilities (even, odd scores)
  bf16x8 sel;         // 0/1 selector: the A operand of the row-sum MFMA
  float c, thr_raw;
  int li, hh;
  uint32_t kb4[4];  // LDS byte address of this lane's K operand reads in the next tile's K
                    // (line_k_rd(lane, j)); advanced one stage per tile
  uint32_t vb2[2];  // ... of its V^T operand reads in this tile's V (line_v_tr(lane, p))

  // LDS read bases start at ring stage 0 (tile 0).
  __device__ __forceinline__ void setup(int lane, float c_, uint32_t ring) {
    li = lane & 31;
    hh = lane >> 5;
#pragma unroll
    for (int j = 0; j < 4; ++j) kb4[j] = ring + 2u * (uint32_t)line_k_rd(lane, j);
    vb2[0] = ring + kVOff + 2u * (uint32_t)line_v_tr(lane, 0);
    vb2[1] = ring + kVOff + 2u * (uint32_t)line_v_tr(lane, 1);
    c = c_;
    thr_raw = kRescaleThreshold / c;
    // Zeros pinned into AGPRs, the file every later MFMA keeps O in.
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int qb = 0; qb < 2; ++qb) {
        o[dt][qb] = f32x16{};
        asm volatile("" : "+a"(o[dt][qb]));
      }
    m_raw[0] = m_raw[1] = -INFINITY;
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
      lsum[qb] = f32x4{};
      asm volatile("" : "+a"(lsum[qb]));
    }
    // Row sums by v_mfma_f32_16x16x32_bf16 with the P^T operand as B: in that
    // shape lane l's 8 values are B[k = 8 (l / 16) + i][n = l % 16], i.e.
    // query n (+16 for odd l / 16) over one half of the chunk's keys. With
    // A[m][k] = 1 where bit 2 of m equals bit 3 of k, D[m][n] sums query n
    // for m % 8 < 4 and query n + 16 otherwise, which puts the row sum of
    // query li = lane % 32 in all four D values of lane `lane`. Column n holds
    // both queries' P, so a NaN in one makes the sum of the other NaN too.
    {
      const bf16 one = (bf16)(((lane & 15) >> 2 & 1) == ((lane >> 4) & 1) ? 1.0f : 0.0f);
#pragma unroll
      for (int i = 0; i < 8; ++i) sel[i] = one;
      asm volatile("" : "+a"(sel));
    }
  }

  // Q^T operands from this wave's 64 staged rows (two 32-row staging areas),
  // kept in AGPRs (the MFMA reads its B operand from either file).
  __device__ __forceinline__ void read_q(const bf16* stage, int lane) {
#pragma unroll
    for (int qb = 0; qb < 2; ++qb)
#pragma unroll
      for (int kk = 0; kk < 8; ++kk) {
        qreg[qb][kk] = staged_operand(stage + qb * 4096, lane, kk);
        asm volatile("" : "+a"(qreg[qb][kk]));
      }
  }

  // K operand pair j = 8 kb + kk (keys 32 kb .., head-dim 16 kk ..) of the K
  // tile at kb4.
  template <int j>
  __device__ __forceinline__ bf16x8 k_op() const {
    constexpr int kb = j >> 3, kk = j & 7;
    return lds_ld16(kb4[kk & 3] + 8192u * (kk >> 2) + 4096u * kb);
  }
  // V^T operand pair pp = 4 c4 + dt (d 32 dt .., keys of chunk c4).
  template <int pp>
  __device__ __forceinline__ bf16x8 v_op() const {
    constexpr int c4 = pp >> 2, dt = pp & 3;
    constexpr uint32_t off = 8192u * (dt >> 1) + 2048u * c4;
    const s16x4 lo = lds_ld8_tr(vb2[dt & 1] + off);
    const s16x4 hi = lds_ld8_tr(vb2[dt & 1] + off + 1024u);
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  }
  // Moves the K / V^T read bases on by `delta` bytes (the next ring stage).
  __device__ __forceinline__ void advance_k(uint32_t delta) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      kb4[j] += delta;
      asm volatile("" : "+v"(kb4[j]));
    }
  }
  __device__ __forceinline__ void advance_v(uint32_t delta) {
    vb2[0] += delta;
    vb2[1] += delta;
    asm volatile("" : "+v"(vb2[0]), "+v"(vb2[1]));
  }

  // Scores of keys at or past klen (tile at key offset kb) to -inf.
  template <int B>
  __device__ __forceinline__ void mask(int kb, int klen) {
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int qb = 0; qb < 2; ++qb)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = kb + 32 * kt + 8 * (r >> 2) + 4 * hh + (r & 3);
          if (key >= klen) s[B][kt][qb][r] = -INFINITY;
        }
  }
  // Max step k (0..15) of S^T buffer B: block kb = k >> 3, query block
  // qb = k & 1, registers 4 ((k >> 1) & 3) .. + 3, into mx[qb].
  template <int B, int k>
  __device__ __forceinline__ void max_step(float (&mx)[2]) const {
    constexpr int kb = k >> 3, qb = k & 1, r0 = 4 * ((k >> 1) & 3);
    const f32x16& a = s[B][kb][qb];
    if constexpr (k < 2) {
      mx[qb] = max2f(max3f(a[r0], a[r0 + 1], a[r0 + 2]), a[r0 + 3]);
    } else {
      mx[qb] = max3f(mx[qb], a[r0], a[r0 + 1]);
      mx[qb] = max3f(mx[qb], a[r0 + 2], a[r0 + 3]);
    }
  }

  // P unit u of S^T buffer B: scores 2 jp, 2 jp + 1 of the P operand (c4, qb),
  // c4 = u >> 3, qb = (u >> 2) & 1, jp = u & 3, and their sum, in three
  // stages one slot apart (fma, exp, pack + sum): the stages of consecutive
  // units share a slot, so no VALU instruction waits on the one before it.
  // fa / fe carry two units' values between the stages.
  template <int B, int u>
  __device__ __forceinline__ void p_fma(const float (&mc)[2], float (&fa)[2][2]) const {
    constexpr int c4 = u >> 3, qb = (u >> 2) & 1, jp = u & 3;
    constexpr int kb = c4 >> 1, r = 8 * (c4 & 1) + 2 * jp;
    fa[u & 1][0] = fmaf(s[B][kb][qb][r], c, -mc[qb]);
    fa[u & 1][1] = fmaf(s[B][kb][qb][r + 1], c, -mc[qb]);
    asm volatile("" : "+v"(fa[u & 1][0]), "+v"(fa[u & 1][1]));
  }
  template <int u>
  __device__ __forceinline__ void p_exp(const float (&fa)[2][2], float (&fe)[2][2]) const {
    fe[u & 1][0] = fast_exp2(fa[u & 1][0]);
    fe[u & 1][1] = fast_exp2(fa[u & 1][1]);
    asm volatile("" : "+v"(fe[u & 1][0]), "+v"(fe[u & 1][1]));
  }
  template <int u, bool FSUM>
  __device__ __forceinline__ void p_pack(const float (&fe)[2][2]) {
    constexpr int c4 = u >> 3, qb = (u >> 2) & 1, jp = u & 3;
    if constexpr (FSUM) {
      lf[qb][0] += fe[u & 1][0];
      lf[qb][1] += fe[u & 1][1];
      asm volatile("" : "+v"(lf[qb][0]), "+v"(lf[qb][1]));
    }
    pb[c4][qb][2 * jp] = (bf16)fe[u & 1][0];
    pb[c4][qb][2 * jp + 1] = (bf16)fe[u & 1][1];
    // Anchored in its slot: left alone, the compiler sinks the P work next to
    // its MFMA users.
    asm volatile("" : "+v"(pb[c4][qb]));
  }
  // Row sums of the P operand (c4, qb) on the matrix pipe (see setup): the
  // VALU alternatives cost the SIMD's vector issue (fp32 adds) or stall the
  // matrix pipe for half an MFMA each (v_dot2c_f32_bf16).
  template <int c4, int qb>
  __device__ __forceinline__ void p_sum() {
    mfma_rowsum(lsum[qb], sel, pb[c4][qb]);
  }

  // S^T of the first tile of the range (no other work to interleave but the
  // DMA's first_slot hook).
  template <int B, class Dma>
  __device__ __forceinline__ void qk_first(const Dma& dma) {
    bf16x8 kq[kKQ];
    static_for<0, 32 + 2 * kKPf>([&](auto G) {
      constexpr int g = decltype(G)::value;
      static_for<0, 16>([&](auto J) {
        constexpr int j = decltype(J)::value;
        if constexpr (kread_slot(j) == g) kq[j % kKQ] = this->template k_op<j>();
      });
      if constexpr (g < 32) {
        constexpr int j = g >> 1, kb = j >> 3, kk = j & 7, qb = g & 1;
        s[B][kb][qb] = mfma32(kq[j % kKQ], qreg[qb][kk], kk == 0 ? f32x16{} : s[B][kb][qb]);
        dma.template first_slot<g>();
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  }

  // Row max of S^T buffer B into mt (no other work).
  template <int B>
  __device__ __forceinline__ void max_plain() {
    float mx[2];
    static_for<0, 16>([&](auto K) { this->template max_step<B, decltype(K)::value>(mx); });
    mt[0] = pair_max(mx[0]);
    mt[1] = pair_max(mx[1]);
  }

  // One tile t of the slot schedule. S^T of tile t is in buffer SB; with
  // NEXT, S^T of tile t+1 (its K one ring stage, dstage bytes, past tile t's)
  // goes to buffer 1 - SB (masked first when its keys end inside it:
  // mask_next) and, with TRACK, its row max to mt. `dma` issues the K/V DMA
  // in the slots (after_slot) and waits for it where the kernel does that in
  // the slots too (before_slot, ahead of the slot's operand reads).
  // Dma::kAnchorS holds the S^T MFMAs in their slots by empty asm statements.
  // FSUM: the fp32 probabilities' row sums too (for an exact LSE).
  template <int SB, bool NEXT, bool TRACK, bool FSUM, class Dma>
  __device__ __forceinline__ void tile(uint32_t dstage, bool mask_next, int kb_next, int klen,
                                       const Dma& dma) {
    constexpr int NB = 1 - SB;
    const float mc[2] = {m_raw[0] * c, m_raw[1] * c};
    if constexpr (NEXT) advance_k(dstage);
    bf16x8 kq[kKQ], vq[kVQ];
    float mx[2];
    float fa[2][2], fe[2][2];
    static_for<0, 64>([&](auto G) {
      constexpr int g = decltype(G)::value;
      if constexpr (NEXT && g == kMaxSlot0) {
        if (mask_next) dma.template mask<NB>(*this, kb_next, klen);
      }
      dma.template before_slot<g, NEXT>();
      // Operand reads.
      if constexpr (NEXT) {
        static_for<0, 16>([&](auto J) {
          constexpr int j = decltype(J)::value;
          if constexpr (kread_slot(j) == g) kq[j % kKQ] = this->template k_op<j>();
        });
      }
      static_for<0, 16>([&](auto P) {
        constexpr int pp = decltype(P)::value;
        if constexpr (vread_slot(pp) == g) vq[pp % kVQ] = this->template v_op<pp>();
      });
      // The slot's MFMA.
      if constexpr (g < 32) {
        if constexpr (NEXT) {
          constexpr int j = g >> 1, kb = j >> 3, kk = j & 7, qb = g & 1;
          s[NB][kb][qb] = mfma32(kq[j % kKQ], qreg[qb][kk], kk == 0 ? f32x16{} : s[NB][kb][qb]);
          if constexpr (Dma::kAnchorS) asm volatile("" : "+v"(s[NB][kb][qb]));
        }
      } else {
        constexpr int op = g - 32, pp = op >> 1, c4 = pp >> 2, dt = pp & 3, qb = op & 1;
        mfma_pv(o[dt][qb], vq[pp % kVQ], pb[c4][qb]);
        if constexpr (dt == 2) this->template p_sum<c4, qb>();
      }

      // P units of tile t, three stages per unit.
      static_for<0, 32>([&](auto U) {
        constexpr int u = decltype(U)::value;
        if constexpr (exp_slot(u) == g) this->template p_fma<SB, u>(mc, fa);
        if constexpr (exp_slot(u) + 1 == g) this->template p_exp<u>(fa, fe);
        if constexpr (exp_slot(u) + 2 == g) this->template p_pack<u, FSUM>(fe);
      });
      // Row max of tile t+1.
      if constexpr (NEXT && TRACK && g >= kMaxSlot0) {
        this->template max_step<NB, g - kMaxSlot0>(mx);
        asm volatile("" : "+v"(mx[0]), "+v"(mx[1]));
      }
      dma.template after_slot<g, NEXT>();
      // The operands of the previous slot's inline-asm MFMA stay allocated to
      // the end of this slot: the compiler does not see that MFMA still
      // reading them and would hand their registers to this slot's VALU
      // results, whose writes would then wait for it.
      if constexpr (g > 32) {
        constexpr int op = g - 33, pp = op >> 1, c4 = pp >> 2, dt = pp & 3, qb = op & 1;
        keep_alive(vq[pp % kVQ]);
        if constexpr (dt == 3) keep_alive(pb[c4][qb]);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    keep_alive(vq[15 % kVQ]);
    keep_alive(pb[3][1]);
    advance_v(dstage);
    if constexpr (NEXT && TRACK) {
      mt[0] = pair_max(mx[0]);
      mt[1] = pair_max(mx[1]);
    }
  }

  // Keeps O in AGPRs up to this point and orders the VALU code that follows
  // after every MFMA that wrote it.
  __device__ __forceinline__ void fence_o() {
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 3"
                 : "+a"(o[0][0]), "+a"(o[1][0]), "+a"(o[2][0]), "+a"(o[3][0]), "+a"(o[0][1]),
                   "+a"(o[1][1]), "+a"(o[2][1]), "+a"(o[3][1]), "+a"(lsum[0]), "+a"(lsum[1]));
  }

  // Lazy rescale for the next tile's max mt: m is raised (and O and l scaled
  // down) only where mt exceeds it by more than thr_raw.
  template <bool FSUM>
  __device__ __forceinline__ void update_max() {
    const bool n0 = mt[0] > m_raw[0] + thr_raw;
    const bool n1 = mt[1] > m_raw[1] + thr_raw;
    if (__builtin_amdgcn_ballot_w64(n0 || n1)) {
      const float mn0 = n0 ? mt[0] : m_raw[0];
      const float mn1 = n1 ? mt[1] : m_raw[1];
      const float a0 = fast_exp2((m_raw[0] - mn0) * c);
      const float a1 = fast_exp2((m_raw[1] - mn1) * c);
      fence_o();
      // One accumulator block at a time, pinned back into AGPRs: otherwise the
      // compiler reads all 128 values into VGPRs first.
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) {
#pragma unroll
        for (int r = 0; r < 16; ++r) o[dt][0][r] *= a0;
        asm volatile("" : "+a"(o[dt][0]));
#pragma unroll
        for (int r = 0; r < 16; ++r) o[dt][1][r] *= a1;
        asm volatile("" : "+a"(o[dt][1]));
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        lsum[0][r] *= a0;
        lsum[1][r] *= a1;
      }
      asm volatile("" : "+a"(lsum[0]), "+a"(lsum[1]));
      if constexpr (FSUM) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          lf[0][i] *= a0;
          lf[1][i] *= a1;
        }
      }
      m_raw[0] = mn0;
      m_raw[1] = mn1;
    }
  }

  // After a pass that kept every row's first-tile max as m (no per-tile max,
  // no rescale): whether every row sum is at most 2^64 (so every p was
  // finite and 1/l is a normal number) and every O^T accumulator finite.
  // Then the result is the one a running max gives, up to fp32 rounding: m
  // only sets the exponent range. Reads O, so after fence_o().
  __device__ __forceinline__ bool sums_in_range() const {
    float mo = 0.f;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int qb = 0; qb < 2; ++qb)
#pragma unroll
        for (int r = 0; r < 16; r += 2) mo = max3abs(mo, o[dt][qb][r], o[dt][qb][r + 1]);
    return lsum[0][0] <= 0x1p64f && lsum[1][0] <= 0x1p64f && mo <= 0x1.fffffep127f;
  }

  // O (or the range's partial O) of query block qb: O / l, optional padding
  // correction, bf16, out through the 8 KB staging area `stage` (tile_io.h
  // row staging, 4 whole 256-byte rows per store); LSE in fp32.
  template <int qb>
  __device__ __forceinline__ float finish(float pad_ln, bool pad, bf16* obase, int64_t ors,
                                          int orow0, int onrows, int lane, bf16* stage) const {
    const float l_tot = lsum[qb][0];
    const bool any = l_tot > 0.f;
    const float lse = any ? (m_raw[qb] * c + __log2f(l_tot)) * kLn2 : -INFINITY;
    float scale = any ? 1.0f / l_tot : 0.f;
    if (pad) scale *= 1.0f / (1.0f + expf(pad_ln - lse));
    const f32x16 ob[4] = {o[0][qb], o[1][qb], o[2][qb], o[3][qb]};
    stage_acc_rows(ob, scale, lane, stage);
    stage_rows_out(obase, ors, orow0, onrows, lane, stage);
    return lse;
  }
};

}  // namespace aa
