// dQ of the attention backward for short query ranges (gfx950): one workgroup
// = 64 queries of one (batch, head), its keys split over the 4 waves inside
// the workgroup, as the forward does it (attn_fwd_ks.hip).
//
// Why: dq_kernel takes 256 queries per workgroup, so 1024 tokens x 16 heads
// are 64 workgroups on 256 CUs, and a key split over workgroups would move
// fp32 partials of four times dQ's size through memory. Here wave w takes the
// 32-key blocks w, w + 4, ..., all waves hold the same 64 queries' Q^T and
// dO^T in registers, and the four fp32 partial dQ^T are summed in wave order
// through LDS: deterministic, no workspace, 256 workgroups for that call.
//
// Per key block j of a wave, 48 slots of one MFMA, with the block's VALU work
// dealt to fixed slots (sched_barrier), as in the other one-wave kernels:
//   slots  0-15: dP^T - D = V dO^T of block j+1 | dZ^T of block j:
//   slots 16-31: S^T = K Q^T of block j+1       |   fma, exp, mul, pack
//   slots 32-47: dQ^T += K^T dZ^T of block j    | (slots 0-38)
// K blocks live in a ring of three 8 KB places (rows of j+1, transposed reads
// of j, and j+2 on its way), V blocks in a ring of two: 40 KB per wave, the
// CU's whole LDS for four. Each place is refilled as soon as its last operand
// is read, by one DMA instruction per odd slot: V of block j+3 in slots 17-31
// (8), the first 16 keys of K of block j+3 in slots 41-47 (4) and the last 16
// of block j+2 in slots 1-7 (4). They then have 50-70 slots (about 1 us) to
// arrive, and the waits ahead of the first V read (all but the 20 youngest)
// and the first K read (16) cover exactly the loads up to those blocks.
#include <type_traits>

#include "attn_bwd.h"
#include "tile_io.h"

namespace aa {
namespace bwd {
namespace dqks {

constexpr int kWaves = 4;
constexpr int kKeys = 32;                                  // keys per block
constexpr uint32_t kBlock = kKeys * kD * sizeof(bf16);     // 8 KB
constexpr uint32_t kVRing = 3 * kBlock;                    // V ring past the K ring
constexpr uint32_t kWaveBytes = 5 * kBlock;                // 40 KB

template <int n>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(n) : "memory");
}
__device__ __forceinline__ void mfma_acc(f32x16& acc, bf16x8 a, bf16x8 b) {
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}
__device__ __forceinline__ void keep_alive(bf16x8 v) { asm volatile("" ::"v"(v)); }

// Unit u of a block: scores 2 jp, 2 jp + 1 of the dZ operand (c, qb), c =
// u >> 3, qb = (u >> 2) & 1, jp = u & 3; three stages from slot unit_slot(u).
constexpr int unit_slot(int u) { return (12 * u) / 5; }
// Operands are read two pairs of slots ahead of their MFMAs.
constexpr int kPf = 2, kRowQ = kPf + 1, kTrQ = kPf + 2;
constexpr int vrow_slot(int j) { return j < kPf ? 0 : 2 * (j - kPf); }
constexpr int krow_slot(int j) { return 16 + 2 * (j - kPf); }
constexpr int ktr_slot(int j) { return 32 + 2 * (j - kPf); }

// A block as 8 KB of dual line tile (tile_io.h) with 4 row blocks per d half:
// 1 KB block 4 dh + row / 8.
struct BlockDma {
  uint32_t ko[4], vo[4];    // per-lane byte offsets of the 8-row blocks
  const bf16 *kt, *vt;      // first rows of the K block (its last 16 keys) and V block being
                            // fetched, and of the K block whose first 16 keys are
  const bf16* ka;
  uint32_t kdst, vdst, kadst;  // LDS byte addresses of their places

  // Rows at or past Sk are never fetched: fewer than 32 keys re-read the last
  // one, more have no block that reaches past them (row_of in the kernel).
  __device__ __forceinline__ void setup(const Params& p, int lane) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = min(8 * i + (lane >> 3), p.Sk - 1), col = 8 * dual_chunk(lane, i & 1);
      ko[i] = (uint32_t)(r * p.s_k[1] + col) * 2u;
      vo[i] = (uint32_t)(r * p.s_v[1] + col) * 2u;
    }
  }
  template <int i>
  __device__ __forceinline__ void issue_k() const {
    dma16_sva_off<128 * (i >> 2), 1024 * i>(kt, ko[i & 3], kdst);
  }
  // Instruction i (0-3) of the first 16 keys of the block at ka; of the last
  // 16 of the block at kt.
  template <int i>
  __device__ __forceinline__ void issue_ka() const {
    constexpr int m = (i & 1) + 4 * (i >> 1);
    dma16_sva_off<128 * (m >> 2), 1024 * m>(ka, ko[m & 3], kadst);
  }
  template <int i>
  __device__ __forceinline__ void issue_kb() const {
    this->template issue_k<2 + (i & 1) + 4 * (i >> 1)>();
  }
  template <int i>
  __device__ __forceinline__ void issue_v() const {
    dma16_sva_off<128 * (i >> 2), 1024 * i>(vt, vo[i & 3], vdst);
  }
  __device__ __forceinline__ void all_k() const {
    static_for<0, 8>([&](auto I) { this->template issue_k<decltype(I)::value>(); });
  }
  __device__ __forceinline__ void all_v() const {
    static_for<0, 8>([&](auto I) { this->template issue_v<decltype(I)::value>(); });
  }
};

struct DqWave {
  bf16x8 qop[2][8], dop[2][8];  // Q^T (AGPRs) / dO^T (qb, kk): [query 32 qb + li][16 kk + 8 hh + ..]
  f32x16 dq[4][2];              // dQ^T (dt, qb): d = 32 dt + rows, query 32 qb + li; AGPRs
  f32x16 s[2][2], dp[2][2];     // S^T, dP^T - D (buffer, qb): keys of the block, query 32 qb + li
  bf16x8 zb[2][2];              // dZ^T (c, qb): keys 16 c + .. in accumulator order
  float lse2[2];                // lse * log2(e) of query 32 qb + li
  f32x16 nd[2];                 // its -D in every element: where dP^T - D starts
  float c;
  int li, hh;
  uint32_t krd[4], vrd[4];      // LDS byte addresses of the next block's K / V row operands
  uint32_t ktr[4];              // ... of this block's K transposed operands

  template <int j>
  __device__ __forceinline__ bf16x8 k_row() const {
    return lds_ld16(krd[j & 3] + 4096u * (j >> 2));
  }
  template <int j>
  __device__ __forceinline__ bf16x8 v_row() const {
    return lds_ld16(vrd[j & 3] + 4096u * (j >> 2));
  }
  // K^T operand j = 4 c + dt.
  template <int j>
  __device__ __forceinline__ bf16x8 k_tr() const {
    constexpr int c4 = j >> 2, dt = j & 3;
    constexpr uint32_t off = 4096u * (dt >> 1) + 2048u * c4;
    const s16x4 lo = lds_ld8_tr(ktr[2 * (dt & 1)] + off);
    const s16x4 hi = lds_ld8_tr(ktr[2 * (dt & 1) + 1] + off + 1024u);
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  }
  // Move the read bases on by `dk`, `dv` bytes (the next places of the rings).
  __device__ __forceinline__ void advance_rows(uint32_t dk, uint32_t dv) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      krd[i] += dk;
      vrd[i] += dv;
      asm volatile("" : "+v"(krd[i]), "+v"(vrd[i]));
    }
  }
  __device__ __forceinline__ void advance_tr(uint32_t dk) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      ktr[i] += dk;
      asm volatile("" : "+v"(ktr[i]));
    }
  }

  // MFMA g (0-31) of dP^T - D and S^T into buffer B.
  template <int B, int g>
  __device__ __forceinline__ void x_mfma(bf16x8 a) {
    constexpr int kk = (g & 15) >> 1, qb = g & 1;
    if constexpr (g < 16) dp[B][qb] = mfma32(a, dop[qb][kk], kk == 0 ? nd[qb] : dp[B][qb]);
    else s[B][qb] = mfma32(a, qop[qb][kk], kk == 0 ? f32x16{} : s[B][qb]);
  }

  // Scores of keys outside [lo, Sk) (block at key row kb) to -inf: dZ = 0.
  template <int B>
  __device__ __forceinline__ void mask(int kb, int lo, int Sk) {
#pragma unroll
    for (int qb = 0; qb < 2; ++qb)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = kb + 8 * (r >> 2) + 4 * hh + (r & 3);
        if (key < lo || key >= Sk) s[B][qb][r] = -INFINITY;
      }
  }

  // S^T and dP^T - D of the wave's first block (no other work).
  template <int B>
  __device__ __forceinline__ void first() {
    bf16x8 rq[kRowQ];
    static_for<0, 32>([&](auto G) {
      constexpr int g = decltype(G)::value;
      static_for<0, 8>([&](auto J) {
        constexpr int j = decltype(J)::value;
        if constexpr (vrow_slot(j) == g) rq[j % kRowQ] = this->template v_row<j>();
        if constexpr (krow_slot(j) == g) rq[(8 + j) % kRowQ] = this->template k_row<j>();
      });
      this->template x_mfma<B, g>(rq[(g >> 1) % kRowQ]);
      __builtin_amdgcn_sched_barrier(0);
    });
  }

  // Block j: dZ^T and dQ^T of block j (its S^T, dP^T - D in buffer SB) and,
  // with NEXT, those of block j+1 into the other buffer.
  template <int SB, bool NEXT>
  __device__ __forceinline__ void block(bool mask_next, int kb_next, int lo_next, int Sk,
                                        const BlockDma& dma) {
    constexpr int NB = 1 - SB;
    bf16x8 rq[kRowQ], tq[kTrQ];
    float fa[2][2], fe[2][2];
    static_for<0, 48>([&](auto G) {
      constexpr int g = decltype(G)::value;
      if constexpr (NEXT && g == krow_slot(0)) wait_vm<16>();  // K of block j+1
      static_for<0, 8>([&](auto J) {
        constexpr int j = decltype(J)::value;
        if constexpr (NEXT && vrow_slot(j) == g) rq[j % kRowQ] = this->template v_row<j>();
        if constexpr (NEXT && krow_slot(j) == g) rq[(8 + j) % kRowQ] = this->template k_row<j>();
        if constexpr (ktr_slot(j) == g) tq[j % kTrQ] = this->template k_tr<j>();
      });
      if constexpr (g < 32) {
        if constexpr (NEXT) {
          this->template x_mfma<NB, g>(rq[(g >> 1) % kRowQ]);
          // Anchored in its slot: left alone, the compiler moves these MFMAs
          // down to where mask and the next block read them, all in a row
          // behind the VALU work that they are meant to cover (backward at
          // 512 x 4096 keys 84 -> 76 us, 2048 tokens 117-119 -> 112-116).
          f32x16& acc = g < 16 ? dp[NB][g & 1] : s[NB][g & 1];
          asm volatile("" : "+v"(acc));
        }
      } else {
        constexpr int op = g - 32, j = op >> 1;
        mfma_acc(dq[j & 3][op & 1], tq[j % kTrQ], zb[j >> 2][op & 1]);
      }
      static_for<0, 16>([&](auto U) {
        constexpr int u = decltype(U)::value;
        constexpr int cz = u >> 3, qb = (u >> 2) & 1, jp = u & 3, r = 8 * cz + 2 * jp;
        if constexpr (unit_slot(u) == g) {
          fa[u & 1][0] = fmaf(s[SB][qb][r], c, -lse2[qb]);
          fa[u & 1][1] = fmaf(s[SB][qb][r + 1], c, -lse2[qb]);
          asm volatile("" : "+v"(fa[u & 1][0]), "+v"(fa[u & 1][1]));
        }
        if constexpr (unit_slot(u) + 1 == g) {
          fe[u & 1][0] = fast_exp2(fa[u & 1][0]);
          fe[u & 1][1] = fast_exp2(fa[u & 1][1]);
          asm volatile("" : "+v"(fe[u & 1][0]), "+v"(fe[u & 1][1]));
        }
        if constexpr (unit_slot(u) + 2 == g) {
          zb[cz][qb][2 * jp] = (bf16)(fe[u & 1][0] * dp[SB][qb][r]);
          zb[cz][qb][2 * jp + 1] = (bf16)(fe[u & 1][1] * dp[SB][qb][r + 1]);
          asm volatile("" : "+v"(zb[cz][qb]));
        }
      });
      if constexpr (NEXT && g == 40) {
        if (mask_next) mask<NB>(kb_next, lo_next, Sk);
      }
      if constexpr (NEXT && (g & 1)) {
        if constexpr (g < 8) dma.template issue_kb<(g >> 1)>();
        if constexpr (g >= 16 && g < 32) dma.template issue_v<((g - 16) >> 1)>();
        if constexpr (g >= 40) dma.template issue_ka<((g - 40) >> 1)>();
      }
      // The operands of the previous slot's inline-asm MFMA stay allocated to
      // the end of this slot: the compiler does not see it still reading them.
      if constexpr (g > 32) {
        constexpr int op = g - 33;
        keep_alive(tq[(op >> 1) % kTrQ]);
        keep_alive(zb[op >> 3][op & 1]);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    keep_alive(tq[7 % kTrQ]);
    keep_alive(zb[1][1]);
  }
};

__global__ __launch_bounds__(kWaves * 64) __attribute__((amdgpu_waves_per_eu(1, 1)))
void dq_ks_kernel(Params p, int first_item, int nqitem, int total_blocks) {
  __shared__ __attribute__((aligned(1024))) uint8_t lds[kWaves * kWaveBytes];

  // A quarter of one of dq_kernel's items of 256 queries.
  const int logical = xcd_remap(blockIdx.x, total_blocks);
  const int item = first_item + logical / 4;
  const int bh = item / nqitem;
  const int qblk = 4 * (item - bh * nqitem) + (logical & 3);
  if (qblk >= p.ntq) return;
  const int b = bh / p.H, h = bh - b * p.H;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int li = lane & 31, hh = lane >> 5;
  const int qrow0 = qblk * kT;

  // Q, dO and O rows (64 each) into places of the rings that the first blocks
  // leave free: the third K place of waves 0-1, 2-3 and the second V place of
  // waves 0-1, as areas of 32 rows (row staging, tile_io.h). Each wave moves
  // 16 rows of each tensor.
  auto area = [&](int w, uint32_t off) { return reinterpret_cast<bf16*>(lds + w * kWaveBytes + off); };
  auto stage_in = [&](const bf16* base, int64_t rs, bf16* a0, bf16* a1) {
    bf16* a = (wave & 2) ? a1 : a0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 16 * (wave & 1) + 4 * i + (lane >> 4);
      const int row = min(qrow0 + 32 * (wave >> 1) + r, p.Sq - 1);
      dma16(base + (int64_t)row * rs + 8 * ((lane & 15) ^ (r & 15)), a + (16 * (wave & 1) + 4 * i) * 128);
    }
  };
  bf16* aq[2] = {area(0, 2 * kBlock), area(1, 2 * kBlock)};
  bf16* ado[2] = {area(2, 2 * kBlock), area(3, 2 * kBlock)};
  bf16* ao[2] = {area(0, kVRing + kBlock), area(1, kVRing + kBlock)};
  stage_in(p.q + b * p.s_q[0] + h * p.s_q[2], p.s_q[1], aq[0], aq[1]);
  stage_in(p.dout + b * p.s_do[0] + h * p.s_do[2], p.s_do[1], ado[0], ado[1]);
  stage_in(p.o + b * p.s_o[0] + h * p.s_o[2], p.s_o[1], ao[0], ao[1]);

  // The wave's i-th block is key block wave + 4 i; one that would reach past
  // Sk is moved back to end there, its keys below lo_of (counted by the
  // blocks before it) masked. Past the wave's last, the last one is fetched
  // again into places that nothing reads.
  const int nblk = (p.Sk + kKeys - 1) / kKeys;
  const int n = (nblk - wave + kWaves - 1) / kWaves;  // 0 if the wave has none
  auto lo_of = [&](int i) { return (wave + kWaves * i) * kKeys; };
  auto row_of = [&](int i) { return min(lo_of(i), max(p.Sk - kKeys, 0)); };
  const bf16* kp = p.k + b * p.s_k[0] + h * p.s_k[2];
  const bf16* vp = p.v + b * p.s_v[0] + h * p.s_v[2];
  const uint32_t mine = lds_addr(lds) + (uint32_t)wave * kWaveBytes;
  BlockDma dma;
  dma.setup(p, lane);
  auto k_job = [&](int i) {
    dma.kt = kp + (int64_t)row_of(min(i, n - 1)) * p.s_k[1];
    dma.kdst = mine + (uint32_t)(i % 3) * kBlock;
  };
  auto ka_job = [&](int i) {
    dma.ka = kp + (int64_t)row_of(min(i, n - 1)) * p.s_k[1];
    dma.kadst = mine + (uint32_t)(i % 3) * kBlock;
  };
  auto v_job = [&](int i) {
    dma.vt = vp + (int64_t)row_of(min(i, n - 1)) * p.s_v[1];
    dma.vdst = mine + kVRing + (uint32_t)(i & 1) * kBlock;
  };
  if (n > 0) {
    k_job(0);
    dma.all_k();
    v_job(0);
    dma.all_v();
    k_job(1);
    dma.all_k();
    wait_vm<8>();  // all but K of block 1
  } else {
    wait_dma();
  }
  __syncthreads();

  DqWave w;
  w.li = li;
  w.hh = hh;
  w.c = p.c;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    w.krd[j] = mine + 2u * (uint32_t)dual_row_rd(lane, j);
    w.vrd[j] = w.krd[j] + kVRing;
    w.ktr[j] = mine + 2u * (uint32_t)dual_tr_rd(lane, j >> 1, j & 1);
  }
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
      w.dq[dt][qb] = f32x16{};
      asm volatile("" : "+a"(w.dq[dt][qb]));
    }
  // Operands, and each query's stats: lse2 = lse log2(e) and -D, D =
  // rowsum(dO o O) (this lane's 64 values, then the partner lane's half).
  // Queries past Sq: lse2 = +inf (P = 0) and D = 0.
#pragma unroll
  for (int qb = 0; qb < 2; ++qb) {
    const int q = qrow0 + 32 * qb + li;
    float nd = 0.f;
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) {
      w.qop[qb][kk] = staged_operand(aq[qb], lane, kk);
      w.dop[qb][kk] = staged_operand(ado[qb], lane, kk);
      float x[8], y[8];
      unpack8(__builtin_bit_cast(u32x4, staged_operand(ao[qb], lane, kk)), x);
      unpack8(__builtin_bit_cast(u32x4, w.dop[qb][kk]), y);
#pragma unroll
      for (int i = 0; i < 8; ++i) nd = fmaf(y[i], x[i], nd);
      asm volatile("" : "+a"(w.qop[qb][kk]));
    }
    nd = pair_sum(nd);
    nd = q < p.Sq ? -nd : 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) w.nd[qb][r] = nd;
    w.lse2[qb] = q < p.Sq ? p.lse[(int64_t)bh * p.Sq + q] * kLog2e : INFINITY;
  }
  // The record that the dK/dV kernel reads: lse2, -D, zero pad.
  if (wave == 0 && hh == 0) {
    float* st = p.stats + ((int64_t)bh * p.ntq + qblk) * kStat;
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
      st[32 * qb + li] = w.lse2[qb];
      st[kT + 32 * qb + li] = w.nd[qb][0];
      st[2 * kT + 32 * qb + li] = 0.f;
      st[3 * kT + 32 * qb + li] = 0.f;
    }
  }
  // The record's stores and the lse loads leave the vmcnt counts to the DMA.
  wait_dma();
  __syncthreads();  // every wave has read the staged rows

  if (n > 0) {
    v_job(1);
    dma.all_v();
    const int b0 = (n - 1) & 1;  // the last block's S^T is in buffer 0
    const bool m0 = lo_of(0) + kKeys > p.Sk;
    if (b0) {
      w.first<1>();
      if (m0) w.mask<1>(row_of(0), lo_of(0), p.Sk);
    } else {
      w.first<0>();
      if (m0) w.mask<0>(row_of(0), lo_of(0), p.Sk);
    }
    v_job(2);
    dma.all_v();
    ka_job(2);
    static_for<0, 4>([&](auto I) { dma.template issue_ka<decltype(I)::value>(); });
    // Once as the blocks' own counts do not hold yet: all but those 12, that
    // is K and V of block 1.
    wait_vm<12>();

    auto run = [&](auto sb, auto next, int i) {
      constexpr int SB = decltype(sb)::value;
      constexpr bool NEXT = decltype(next)::value;
      if constexpr (NEXT) {
        wait_vm<20>();  // V of block i + 1
        w.advance_rows((i + 1) % 3 == 0 ? 0u - 2u * kBlock : kBlock, (i + 1) & 1 ? kBlock : 0u - kBlock);
        k_job(i + 2);
        ka_job(i + 3);
        v_job(i + 3);
      }
      const int lo = lo_of(i + 1);
      w.block<SB, NEXT>(lo + kKeys > p.Sk, row_of(i + 1), lo, p.Sk, dma);
      w.advance_tr((i + 1) % 3 == 0 ? 0u - 2u * kBlock : kBlock);
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
  // Keeps dQ in AGPRs up to here and orders the reads after its MFMAs.
  asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 3"
               : "+a"(w.dq[0][0]), "+a"(w.dq[1][0]), "+a"(w.dq[2][0]), "+a"(w.dq[3][0]),
                 "+a"(w.dq[0][1]), "+a"(w.dq[1][1]), "+a"(w.dq[2][1]), "+a"(w.dq[3][1]));
  __syncthreads();  // every wave is done with its rings

  // Sum over the waves in order: wave d takes head-dims 32 d .. 32 d + 31.
  // Block (dt, source wave, qb, rq) of 1 KB: one float4 per lane.
  f32x4* xch = reinterpret_cast<f32x4*>(lds);
  bf16* stage = reinterpret_cast<bf16*>(lds + 128 * 1024);
  auto at = [&](int dt, int src, int qb, int rq) { return (((dt * kWaves + src) * 2 + qb) * 4 + rq) * 64 + lane; };
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int qb = 0; qb < 2; ++qb)
#pragma unroll
      for (int rq = 0; rq < 4; ++rq) {
        const f32x16& v = w.dq[dt][qb];
        xch[at(dt, wave, qb, rq)] = f32x4{v[4 * rq], v[4 * rq + 1], v[4 * rq + 2], v[4 * rq + 3]};
      }
  __syncthreads();
#pragma unroll
  for (int qb = 0; qb < 2; ++qb)
#pragma unroll
    for (int rq = 0; rq < 4; ++rq) {
      f32x4 v = xch[at(wave, 0, qb, rq)];
#pragma unroll
      for (int src = 1; src < kWaves; ++src) v += xch[at(wave, src, qb, rq)];
      const u32x2 o2 = {pack_bf16(v[0] * p.scale, v[1] * p.scale), pack_bf16(v[2] * p.scale, v[3] * p.scale)};
      *reinterpret_cast<u32x2*>(stage + qb * 4096 + stage_at(li, 4 * wave + rq) + 4 * hh) = o2;
    }
  __syncthreads();
  bf16* ob = p.dq + b * p.s_dq[0] + h * p.s_dq[2];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 16 * wave + 4 * i + (lane >> 4), cc = lane & 15;
    const u32x4 v = *reinterpret_cast<const u32x4*>(stage + (r >> 5) * 4096 + stage_at(r & 31, cc));
    if (qrow0 + r < p.Sq) st16_nt(ob + (int64_t)(qrow0 + r) * p.s_dq[1] + 8 * cc, v);
  }
}

}  // namespace dqks

void launch_dq_ks(const Params& p, int first_item, int items, int nqitem, hipStream_t stream) {
  dqks::dq_ks_kernel<<<dim3((unsigned)(4 * items)), dqks::kWaves * 64, 0, stream>>>(p, first_item, nqitem,
                                                                                  4 * items);
}

}  // namespace bwd
}  // namespace aa
