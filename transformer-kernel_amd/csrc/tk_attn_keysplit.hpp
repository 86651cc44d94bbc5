// Attention for launches that leave most of the chip idle: one workgroup per 32
// query rows, whose NW waves take every NW-th key tile each and merge their
// (row max, row sum, O) at the end.
//
// With few heads and short sequences the other kernels' workgroups of 128 or 256
// query rows are fewer than the 256 CUs, and each walks its key tiles as one
// serial chain of copy, S = Q.K^T, softmax and P.V latencies.  Here there are 4 to
// 8 times the workgroups and a chain is an NW-th as long; in exchange every 32
// rows read K and V from L2 again.
//
// A wave's tiles are its own: K and V slots in LDS that no other wave touches, so
// the loop has no barrier.  The next K copy goes out when the current one's
// fragments have been read, the next V copy after P.V; each is waited for (vmcnt)
// where it is first read.
#pragma once
#include "tk_attn_tile.hpp"

namespace tk {
namespace {

// s_waitcnt lgkmcnt(0): this wave's LDS reads have returned.
__device__ __forceinline__ void wait_lds_reads() {
  __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (0 << 8) | (3 << 14));
}

template <int HD, int NW, bool CAUSAL, bool KMASK, typename Args>
__device__ __forceinline__ void keysplit_body(const Args& p) {
  constexpr int BN = HD <= 128 ? 64 : 32;  // keys per tile
  constexpr int NB = BN / 32;              // 32-key blocks of S^T
  constexpr int RB = HD * 2;              // tile row bytes
  constexpr int CPR = RB / 16;            // 16-byte chunks per row
  constexpr int TILE = BN * RB;           // bytes per K or V tile
  constexpr int COPIES = TILE / 1024;     // 1 KB copies per tile
  constexpr int RPC = 1024 / RB;          // tile rows per copy
  constexpr int DB = (HD + 31) / 32;      // 32-row blocks of the O^T accumulator
  constexpr int KSTEPS = HD / 16;
  constexpr int SLOT = 2 * TILE;          // a wave's K and V
  constexpr int CHUNKS = 4 * DB;          // 4-register pieces of O
  static_assert(HD >= 32 && COPIES < 64 && (CHUNKS % NW == 0 || CHUNKS <= NW), "whole chunks per wave");
  static_assert(CHUNKS * 1024 <= SLOT, "a wave's O fits its slots");
  __shared__ __attribute__((aligned(16))) char smem[NW * SLOT];
  __shared__ float row_m[NW][32], row_l[NW][32];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 5;
  const int BH = p.B * p.H;
  const int n_qt = (p.S + 31) / 32;
  const int id = blockIdx.x;
  const int qt = CAUSAL ? n_qt - 1 - id / BH : id / BH;  // longest first; a head's tiles on one XCD if 8 | B*H
  const int bh = id % BH, b = bh / p.H, h = bh % p.H;
  const int q0 = qt * 32, my_row = q0 + (lane & 31);
  const f16* kb = p.k + b * p.ks[0] + h * p.ks[1];
  const f16* vb = p.v + b * p.vs[0] + h * p.vs[1];
  const uint8_t* kvb = KMASK ? p.kv + b * p.kvs : nullptr;
  char* ks_ = smem + wave * SLOT;
  char* vs_ = ks_ + TILE;
  const uint32_t k_lds = (uint32_t)(size_t)(lds_char*)ks_, v_lds = k_lds + TILE;

  const int kv_end = CAUSAL ? min(p.S, q0 + 32) : p.S;
  const int n_kt = (kv_end + BN - 1) / BN;

  // Lane l of copy c fills physical chunk l % CPR of row c * RPC + l / CPR and fetches
  // the logical chunk that the swizzle keeps there; rows past S re-read row S - 1
  // (their scores are masked).
  auto copy = [&](const f16* base, int64_t rs, int j, uint32_t dst, bool is_v) {
#pragma unroll
    for (int c = 0; c < COPIES; ++c) {
      const int row = c * RPC + lane / CPR, phys = lane % CPR;
      const int chunk = is_v ? phys ^ vswz<RB>(row) : (swz_off<RB>(row, phys) - row * RB) >> 4;
      dma16(base + (int64_t)min(j * BN + row, p.S - 1) * rs + chunk * 8, dst + c * 1024);
    }
  };

  f16x8 qf[KSTEPS];
  {
    const f16* qr = p.q + b * p.qs[0] + h * p.qs[1] + (int64_t)min(my_row, p.S - 1) * p.qs[2] + g * 8;
#pragma unroll
    for (int kk = 0; kk < KSTEPS; ++kk) qf[kk] = *reinterpret_cast<const f16x8*>(qr + kk * 16);
  }
  if (wave < n_kt) {
    copy(kb, p.ks[2], wave, k_lds, false);
    copy(vb, p.vs[2], wave, v_lds, true);
  }

  int v_rd[2][DB];  // transposed V reads, as attend_one_tile
  {
    const int tq = lane >> 4, ts = lane & 15;
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int d = 0; d < DB; ++d) {
        const int row = 8 * r + 4 * (tq >> 1) + (ts >> 2);
        const int col = 32 * d + 16 * (tq & 1) + 4 * (ts & 3);
        v_rd[r][d] = row * RB + (((col >> 3) ^ vswz<RB>(row)) << 4) + (col & 7) * 2;
      }
  }

  f32x16 acc_o[DB];
#pragma unroll
  for (int d = 0; d < DB; ++d) acc_o[d] = f32x16{};
  float m_run = -INFINITY;  // running max of scale * log2e * s
  float l_run = 0.f;        // this lane's keys
  const float cs = p.scale_log2;

  for (int kt = wave; kt < n_kt; kt += NW) {
    const bool more = kt + NW < n_kt;
    int kbyte = 1;
    if (KMASK) kbyte = kvb[min(kt * BN + lane, p.S - 1)];
    wait_vmcnt<COPIES>();  // all but V's copies: K has landed
    asm volatile("" ::: "memory");
    f32x16 s[NB];
#pragma unroll
    for (int c = 0; c < NB * KSTEPS; ++c) {
      const int kb2 = c / KSTEPS, kk = c % KSTEPS;
      const f16x8 kf = *reinterpret_cast<const f16x8*>(ks_ + swz_off<RB>(kb2 * 32 + (lane & 31), 2 * kk + g));
      s[kb2] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qf[kk], kk == 0 ? f32x16{} : s[kb2], 0, 0, 0);
    }
    // every K fragment is in registers: the slot may be refilled
    asm volatile("" ::: "memory");
    wait_lds_reads();
    // (a validity byte is waited for here, before the copies that may stay in flight)
    const uint64_t kbits = (KMASK ? (uint64_t)__ballot(kbyte != 0) : ~0ull) >> (4 * g);
    if (more) copy(kb, p.ks[2], kt + NW, k_lds, false);

    const int k0 = kt * BN;
    float mx = -INFINITY;
    if (KMASK || k0 + BN > p.S || (CAUSAL && k0 + BN - 1 > q0)) {
#pragma unroll
      for (int e = 0; e < 16 * NB; ++e) {
        const int j = (e >> 4) * 32 + 8 * ((e & 15) >> 2) + (e & 3), key = k0 + j + 4 * g;
        if (key >= p.S || (CAUSAL && key > my_row) || (KMASK && ((kbits >> j) & 1) == 0))
          s[e >> 4][e & 15] = -INFINITY;
      }
    }
#pragma unroll
    for (int e = 0; e < 16 * NB; ++e) mx = fmaxf(mx, s[e >> 4][e & 15]);
    const float m_new = fmaxf(m_run, pair_max(mx) * cs);  // cs > 0
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_use);
    m_run = m_new;
    f16x8 pf[2 * NB];
    float ls = 0.f;
#pragma unroll
    for (int e = 0; e < 16 * NB; ++e) {
      const float pe = __builtin_amdgcn_exp2f(fmaf(s[e >> 4][e & 15], cs, -m_use));
      pf[e >> 3][e & 7] = (f16)pe;
      ls += pe;
    }
    l_run = l_run * alpha + ls;
#pragma unroll
    for (int d = 0; d < DB; ++d)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc_o[d][r] *= alpha;

    if (more) wait_vmcnt<COPIES>();  // all but the next K's copies
    else wait_vmcnt<0>();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int c = 0; c < 2 * NB * DB; ++c) {
      const int t = c / DB, d = c % DB;
      const lds_char* base = (const lds_char*)(vs_ + t * 16 * RB);
      const tr_f16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4f16((lds_tr_f16x4*)(base + v_rd[0][d]));
      const tr_f16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4f16((lds_tr_f16x4*)(base + v_rd[1][d]));
      const f16x8 vf = __builtin_shufflevector(__builtin_bit_cast(f16x4, lo), __builtin_bit_cast(f16x4, hi), 0, 1, 2,
                                               3, 4, 5, 6, 7);
      acc_o[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, pf[t], acc_o[d], 0, 0, 0);
    }
    asm volatile("" ::: "memory");
    wait_lds_reads();
    if (more) copy(vb, p.vs[2], kt + NW, v_lds, true);
  }

  // ---- merge: O rescaled to the rows' common max, sums in wave order ----
  // A wave writes its O (CHUNKS of 64 lanes x 16 bytes) into its own slots.
  asm volatile("" ::: "memory");
  l_run = pair_sum(l_run);
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const f32x16& o = acc_o[c / 4];
    const int q = c % 4;
    *reinterpret_cast<f32x4*>(ks_ + c * 1024 + lane * 16) = f32x4{o[4 * q], o[4 * q + 1], o[4 * q + 2], o[4 * q + 3]};
  }
  if (g == 0) {
    row_m[wave][lane] = m_run;
    row_l[wave][lane] = l_run;
  }
  __syncthreads();
  float f[NW], m_all = -INFINITY, l_all = 0.f;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    f[w] = row_m[w][lane & 31];
    m_all = fmaxf(m_all, f[w]);
  }
  const float m_ref = m_all == -INFINITY ? 0.f : m_all;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    f[w] = __builtin_amdgcn_exp2f(f[w] - m_ref);
    l_all += f[w] * row_l[w][lane & 31];
  }
  const float inv = 1.0f / l_all;
  f16* orow = p.o + b * p.os[0] + h * p.os[1] + (int64_t)my_row * p.os[2];
#pragma unroll
  for (int c0 = 0; c0 < CHUNKS; c0 += NW) {
    const int c = c0 + wave;
    if (CHUNKS % NW != 0 && c >= CHUNKS) break;
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(smem + w * SLOT + c * 1024 + lane * 16);
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] += f[w] * v[e];
    }
    if (my_row < p.S)
      *reinterpret_cast<f16x4*>(orow + (c / 4) * 32 + 8 * (c % 4) + 4 * g) =
          f16x4{(f16)(o[0] * inv), (f16)(o[1] * inv), (f16)(o[2] * inv), (f16)(o[3] * inv)};
  }
}

}  // namespace
}  // namespace tk
