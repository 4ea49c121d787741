// Flash-attention forward for short query ranges, head_dim 128 (gfx950): one
// workgroup = 64 queries of one (batch, head), its keys split over the 4
// waves inside the workgroup.
//
// Why: with 256 queries per work item a small image fills a fraction of the
// chip (1024 tokens x 16 heads: 64 items on 256 CUs) unless the keys are
// split over workgroups, and then the partial O rows go through memory and a
// second launch merges them. Here the split stays inside the workgroup: wave
// w takes key tiles w, w + 4, ..., all four hold the same 64 queries, and the
// four partial results are merged in fp32 through LDS. 1024 tokens x 16 heads
// are 256 workgroups, one per CU, with 4 key tiles per wave.
//
// Each wave runs FwdWave's slot schedule on a K tile and a V tile of its own
// (32 KB of LDS per wave), with no barrier between the waves until the merge.
// A tile is streamed into the place of the one before it, a quarter (4 KB, 4
// DMA instructions) as soon as its last operand has been read:
//   slots  8-15, 16-23, 24-31, 32-39: K quarters 0-3 of tile t+2 (quarter
//     2 kb + dh = keys 32 kb .., head-dim half dh, read in slots 8 q .. 8 q + 7)
//   slots 40-47, 48-55, 56-63 and 0-7 of tile t+1: V key chunks 0-3 of tile
//     t+1 (chunk c, read in slots 32 + 8 c .. 32 + 8 c + 7)
// one instruction in every odd slot, 32 per tile. Every quarter then has
// about 56 slots (2000 cycles) to arrive, and a wait for "all but the 22
// youngest" (24 at slot 0) ahead of each quarter's first read covers exactly
// the loads up to it.
#include <cfloat>
#include <type_traits>

#include "attn_fwd_ks.h"
#include "attn_fwd_wave.h"

namespace aa {
namespace ks {

constexpr int kWaves = 4;
constexpr uint32_t kWaveBytes = 2u * kTileElems * sizeof(bf16);  // a wave's K tile, then V tile
constexpr uint32_t kRingBytes = kWaves * kWaveBytes;             // 128 KB
constexpr uint32_t kStageBytes = kKsQueries * kD * sizeof(bf16); // Q rows in, O rows out: 16 KB

template <int n>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(n) : "memory");
}

// One wave's K/V DMA (the hooks of FwdWave::tile).
struct WaveDma {
  // S^T held in its slots: left alone, the compiler moved these MFMAs of a
  // tile down to the mask's branch, all 32 in a row behind the VALU work that
  // they are meant to cover (when added, 1024 tokens 15.1 -> 14.3 us, 512 11.0
  // -> 10.5; with the plain last tile below 14.1 and 10.1).
  static constexpr bool kAnchorS = true;
  const bf16 *kp, *vp;      // the (batch, head)'s K and V
  int64_t ks1, vs1;         // token strides
  uint32_t ko[8], vo[8];    // per-lane byte offsets of the tile's 8-row blocks
  uint32_t lds;             // LDS byte address of the wave's K tile
  const bf16 *kt, *vt, *v3; // first rows of the K tile and V tile (chunks 0-2; 3) being fetched

  // Rows at or past klen are never fetched (V may hold anything there, and 0
  // times a NaN is one): the wave's last tile re-reads its last row past it
  // (rows_k, rows_v from their first fetch on; what follows is that tile again).
  __device__ __forceinline__ void setup(const FwdParams& p, const bf16* k, const bf16* v, int lane,
                                        uint32_t lds_) {
    kp = k;
    vp = v;
    ks1 = p.ks1;
    vs1 = p.vs1;
    rows_k(lane, kBN - 1);
    rows_v<0, 8>(lane, kBN - 1);
    lds = lds_;
  }
  // Row offsets of a tile whose rows past `last` re-read it (V: blocks I .. E - 1).
  __device__ __forceinline__ void rows_k(int lane, int last) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      ko[i] = (uint32_t)(min(8 * i + (lane >> 3), last) * ks1 + 8 * line_k_chunk(lane, i & 1)) * 2u;
  }
  template <int I, int E>
  __device__ __forceinline__ void rows_v(int lane, int last) {
#pragma unroll
    for (int i = I; i < E; ++i)
      vo[i] = (uint32_t)(min(8 * i + (lane >> 3), last) * vs1 + 8 * line_v_chunk(lane)) * 2u;
  }

  // Instruction i (0-3) of K quarter q / V chunk c: 8 rows x 64 d into the
  // line tile's block 8 dh + row / 8.
  template <int q, int i>
  __device__ __forceinline__ void issue_k() const {
    constexpr int kb = q >> 1, dh = q & 1, blk = 4 * kb + i;
    dma16_sva_off<128 * dh, (8 * dh + blk) * 1024>(kt, ko[blk], lds);
  }
  template <int c, int i>
  __device__ __forceinline__ void issue_v() const {
    constexpr int dh = i >> 1, blk = 2 * c + (i & 1);
    dma16_sva_off<128 * dh, kVOff + (8 * dh + blk) * 1024>(c == 3 ? v3 : vt, vo[blk], lds);
  }

  template <int B, class W>
  __device__ __forceinline__ void mask(W& w, int kb, int klen) const { w.template mask<B>(kb, klen); }
  template <int g>
  __device__ __forceinline__ void first_slot() const {
    constexpr int q = (g >> 3) - 1, i = (g & 7) >> 1;
    if constexpr (q >= 0 && (g & 1)) issue_k<q, i>();
  }
  template <int g, bool NEXT>
  __device__ __forceinline__ void before_slot() const {
    if constexpr (NEXT) {
      if constexpr (g == 0) wait_vm<24>();
      if constexpr (g == 4 || g == 12 || g == 20 || g == 28 || g == 36 || g == 44 || g == 52)
        wait_vm<22>();
    } else {
      // The last tile: only V chunk 3 of this tile went out in its slots.
      if constexpr (g == 28) wait_vm<12>();
      if constexpr (g == 36) wait_vm<8>();
      if constexpr (g == 44) wait_vm<4>();
      if constexpr (g == 52) wait_vm<0>();
    }
  }
  template <int g, bool NEXT>
  __device__ __forceinline__ void after_slot() const {
    if constexpr (g & 1) {
      constexpr int grp = g >> 3, i = (g & 7) >> 1;
      if constexpr (grp == 0) issue_v<3, i>();
      else if constexpr (!NEXT) return;
      else if constexpr (grp <= 4) issue_k<grp - 1, i>();
      else issue_v<grp - 5, i>();
    }
  }
};

// The wave's row sum of query 32 qb + lane % 32 again, in plain arithmetic, for
// rows whose sum on the matrix pipe took in another row's NaN or infinity
// (FwdWave::setup; their O did not). From the staged Q rows and K in memory,
// half of the keys per lane of a pair; only runs where a row holds no finite
// numbers.
__device__ __forceinline__ float row_sum_again(const FwdParams& p, const WaveDma& dma, const bf16* stage,
                                               int qb, int lane, int wave, int n, int klen, float m) {
  const bf16* q = stage + qb * 4096;
  const float mc = m * p.c;
  float sum = 0.f;
#pragma unroll 1
  for (int i = 0; i < n; ++i) {
    const int lo = (wave + kWaves * i) * kBN, hi = min(lo + kBN, klen);
#pragma unroll 1
    for (int key = lo + (lane >> 5); key < hi; key += 2) {
      const bf16* kr = dma.kp + (int64_t)key * dma.ks1;
      float s = 0.f;
#pragma unroll 1
      for (int ch = 0; ch < kD / 8; ++ch) {
        float x[8], y[8];
        unpack8(ld16(q + stage_at(lane & 31, ch)), x);
        unpack8(ld16(kr + 8 * ch), y);
#pragma unroll
        for (int e = 0; e < 8; ++e) s = fmaf(x[e], y[e], s);
      }
      sum += round_bf16(fast_exp2(fmaf(s, p.c, -mc)));
    }
  }
  return pair_sum(sum);
}

// LSE: something reads the log-sum-exp (an output, or the padding correction),
// so the fp32 probabilities are summed on the VALU beside the row sums of the
// MFMAs (2-4% of a call: 1024 queries x 512 keys 10.8 -> 11.2 us, x 4096 40.2 ->
// 41.8).
template <bool LSE>
__global__ __launch_bounds__(kWaves * 64) __attribute__((amdgpu_waves_per_eu(1, 1)))
void attn_fwd_ks_kernel(FwdParams p, int nqblk, int total_blocks) {
  __shared__ __attribute__((aligned(1024))) uint8_t lds[kRingBytes + kStageBytes];

  const int item = xcd_remap(blockIdx.x, total_blocks);
  const int qblk = item % nqblk;
  const int bh = item / nqblk;
  const int b = bh / p.H, h = bh - b * p.H;
  const int klen = p.seqused ? min((int)p.seqused[b], p.Sk) : p.Sk;
  const int ntiles = klen > 0 ? (klen + kBN - 1) / kBN : 0;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int li = lane & 31, hh = lane >> 5;
  const int qrow0 = qblk * kKsQueries;

  // Q: 16 rows per wave into the staging area (two 32-row areas of row
  // staging, tile_io.h), read by all waves after the barrier.
  bf16* stage = reinterpret_cast<bf16*>(lds + kRingBytes);
  {
    const bf16* qb = p.q + b * p.qs0 + h * p.qs2;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 16 * wave + 4 * i + (lane >> 4);
      const int row = min(qrow0 + r, p.Sq - 1);
      dma16(qb + (int64_t)row * p.qs1 + 8 * ((lane & 15) ^ (r & 15)), stage + (16 * wave + 4 * i) * 128);
    }
  }

  // The wave's i-th tile is key tile wave + 4 i; `part` is the one that klen
  // ends in (-1: none). A tile past the wave's last re-reads the last one into
  // places that nothing reads again: every tile issues the same number of DMA
  // instructions.
  const int n = (ntiles - wave + kWaves - 1) / kWaves;  // 0 if the wave has none
  auto lo_of = [&](int i) { return (wave + kWaves * i) * kBN; };
  const int part = n > 0 && lo_of(n - 1) + kBN > klen ? n - 1 : -1;
  const int last = klen - lo_of(n - 1) - 1;  // its last row
  WaveDma dma;
  const uint32_t mine = lds_addr(lds) + (uint32_t)wave * kWaveBytes;
  dma.setup(p, p.k + b * p.ks0 + h * p.ks2, p.v + b * p.vs0 + h * p.vs2, lane, mine);
  auto k_tile = [&](int i) {
    dma.kt = dma.kp + (int64_t)lo_of(min(i, n - 1)) * dma.ks1;
    if (i == part) dma.rows_k(lane, last);
  };
  // V chunks 0-2 of tile i; chunk 3.
  auto v_tile = [&](int i) {
    dma.vt = dma.vp + (int64_t)lo_of(min(i, n - 1)) * dma.vs1;
    if (i == part) dma.rows_v<0, 6>(lane, last);
  };
  auto v3_tile = [&](int i) {
    dma.v3 = dma.vp + (int64_t)lo_of(i) * dma.vs1;
    if (i == part) dma.rows_v<6, 8>(lane, last);
  };
  if (n > 0) {
    k_tile(0);
    static_for<0, 16>([&](auto I) {
      constexpr int i = decltype(I)::value;
      dma.template issue_k<(i >> 2), (i & 3)>();
    });
  }

  FwdWave w;
  w.setup(lane, p.c, mine);
  w.lf[0][0] = w.lf[0][1] = w.lf[1][0] = w.lf[1][1] = 0.f;
  wait_dma();
  __syncthreads();
  w.read_q(stage, lane);
  if (n > 0) {
    // As if a tile -1 came before: the K quarters of tile 1, then V chunks
    // 0-2 of tile 0.
    k_tile(1);
    const int b0 = (n - 1) & 1;  // the last tile's S^T is in buffer 0
    const bool m0 = lo_of(0) + kBN > klen;
    if (b0) {
      w.qk_first<1>(dma);
      if (m0) dma.template mask<1>(w, lo_of(0), klen);
    } else {
      w.qk_first<0>(dma);
      if (m0) dma.template mask<0>(w, lo_of(0), klen);
    }
    static_for<0, 4>([&](auto I) { dma.template issue_k<3, decltype(I)::value>(); });
    v_tile(0);
    static_for<0, 12>([&](auto I) {
      constexpr int i = decltype(I)::value;
      dma.template issue_v<(i >> 2), (i & 3)>();
    });
    if (b0) w.max_plain<1>();
    else w.max_plain<0>();
    // Finite also where every score of the wave's first tile is -inf (keys
    // masked by an infinity): s - m would be NaN there, the other waves' keys
    // and this one's later tiles would be lost to it.
    w.m_raw[0] = fmaxf(w.mt[0], -FLT_MAX);
    w.m_raw[1] = fmaxf(w.mt[1], -FLT_MAX);

    auto run = [&](auto sb, auto next, int i) {
      constexpr int SB = decltype(sb)::value;
      constexpr bool NEXT = decltype(next)::value;
      k_tile(i + 2);
      v3_tile(i);
      v_tile(i + 1);
      const int lo = lo_of(i + 1);
      w.tile<SB, NEXT, true, LSE>(0, lo + kBN > klen, lo, klen, dma);
      if constexpr (NEXT) w.update_max<LSE>();
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    int i = 0;
    if (b0) {
      run(I1{}, std::true_type{}, 0);
      i = 1;
    }
    for (; i + 1 < n; i += 2) {
      run(I0{}, std::true_type{}, i);
      run(I1{}, std::true_type{}, i + 1);
    }
    run(I0{}, std::false_type{}, i);
  }
  wait_dma();
  w.fence_o();
  float lsum[2] = {w.lsum[0][0], w.lsum[1][0]};
#pragma unroll
  for (int qb = 0; qb < 2; ++qb) {
    const bool again = !(lsum[qb] <= FLT_MAX);
    if (__builtin_amdgcn_ballot_w64(again)) {
      const float sum = row_sum_again(p, dma, stage, qb, lane, wave, n, klen, w.m_raw[qb]);
      lsum[qb] = again ? sum : lsum[qb];
    }
  }

  // Merge: every wave's (m, l) through the staging area, O^T times its weight
  // in fp32 through the ring. Wave d sums head-dims 32 d .. 32 d + 31 over the
  // waves in order.
  // O is normalised by the sum of the bf16 probabilities that weighted V, the
  // LSE is that of the fp32 ones.
  float* st_m = reinterpret_cast<float*>(stage);       // [wave][64]
  float* st_l = st_m + kWaves * kKsQueries;
  float* st_f = st_l + kWaves * kKsQueries;
  __syncthreads();  // every wave is done with Q and its tiles
#pragma unroll
  for (int qb = 0; qb < 2; ++qb) {
    float lf = 0.f;
    if constexpr (LSE) lf = pair_sum(w.lf[qb][0] + w.lf[qb][1]);
    if (hh == 0) {
      st_m[wave * kKsQueries + 32 * qb + li] = w.m_raw[qb];
      st_l[wave * kKsQueries + 32 * qb + li] = lsum[qb];
      if constexpr (LSE) st_f[wave * kKsQueries + 32 * qb + li] = lf;
    }
  }
  __syncthreads();
  float scale[2], lse[2];
#pragma unroll
  for (int qb = 0; qb < 2; ++qb) {
    float m[kWaves], l[kWaves], mx = -INFINITY;
#pragma unroll
    for (int v = 0; v < kWaves; ++v) {
      m[v] = st_m[v * kKsQueries + 32 * qb + li];
      l[v] = st_l[v * kKsQueries + 32 * qb + li];
      mx = fmaxf(mx, m[v]);
    }
    float sum = 0.f, fsum = 0.f;
#pragma unroll
    for (int v = 0; v < kWaves; ++v) {
      const float a = m[v] > -INFINITY ? fast_exp2((m[v] - mx) * p.c) : 0.f;  // 0: no keys
      sum += l[v] * a;
      if constexpr (LSE) fsum += st_f[v * kKsQueries + 32 * qb + li] * a;
    }
    // No key, or none with a weight: O = 0, LSE = -inf (a NaN sum goes on).
    const bool any = sum != 0.f;
    scale[qb] = any ? fast_exp2((w.m_raw[qb] - mx) * p.c) / sum : 0.f;
    if constexpr (LSE) {
      lse[qb] = any ? (mx * p.c + __log2f(fsum)) * kLn2 : -INFINITY;
      if (p.ln_pad) scale[qb] *= 1.0f / (1.0f + expf(p.ln_pad[b] - lse[qb]));
    }
  }
  // Block (dt, source wave, qb, rq) of 1 KB: one float4 per lane.
  f32x4* xch = reinterpret_cast<f32x4*>(lds);
  auto at = [&](int dt, int src, int qb, int rq) { return (((dt * kWaves + src) * 2 + qb) * 4 + rq) * 64 + lane; };
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int qb = 0; qb < 2; ++qb)
#pragma unroll
      for (int rq = 0; rq < 4; ++rq) {
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = w.o[dt][qb][4 * rq + e] * scale[qb];
        xch[at(dt, wave, qb, rq)] = v;
      }
  __syncthreads();
#pragma unroll
  for (int qb = 0; qb < 2; ++qb)
#pragma unroll
    for (int rq = 0; rq < 4; ++rq) {
      f32x4 v = xch[at(wave, 0, qb, rq)];
#pragma unroll
      for (int src = 1; src < kWaves; ++src) v += xch[at(wave, src, qb, rq)];
      const u32x2 o2 = {pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
      *reinterpret_cast<u32x2*>(stage + qb * 4096 + stage_at(li, 4 * wave + rq) + 4 * hh) = o2;
    }
  __syncthreads();
  // O rows out, 16 per wave.
  bf16* ob = p.o + b * p.os0 + h * p.os2;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 16 * wave + 4 * i + (lane >> 4), c = lane & 15;
    const u32x4 v = *reinterpret_cast<const u32x4*>(stage + (r >> 5) * 4096 + stage_at(r & 31, c));
    if (qrow0 + r < p.Sq) st16_nt(ob + (int64_t)(qrow0 + r) * p.os1 + 8 * c, v);
  }
  if constexpr (LSE) {
    const int q = qrow0 + 32 * wave + li;
    if (p.lse && wave < 2 && hh == 0 && q < p.Sq)
      p.lse[((int64_t)b * p.H + h) * p.Sq + q] = wave ? lse[1] : lse[0];
  }
}

}  // namespace ks

void launch_attn_fwd_ks(const FwdParams& p, int64_t B, hipStream_t stream) {
  const int nqblk = (p.Sq + kKsQueries - 1) / kKsQueries;
  const int total = (int)(B * p.H * nqblk);
  const dim3 grid((unsigned)total);
  if (p.lse || p.ln_pad) ks::attn_fwd_ks_kernel<true><<<grid, ks::kWaves * 64, 0, stream>>>(p, nqblk, total);
  else ks::attn_fwd_ks_kernel<false><<<grid, ks::kWaves * 64, 0, stream>>>(p, nqblk, total);
}

}  // namespace aa
