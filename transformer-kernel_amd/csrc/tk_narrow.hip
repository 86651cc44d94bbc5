// Row-local parts of a block of width 128, fused: everything but attention.
//
//   narrow_qkv_kernel   q|k|v = LN(x) . W_qkv^T + b
//   narrow_tail_kernel  x += ctx . W_o^T + b_o; h = LN2(x);
//                       x += gelu(h . W_1^T + b_1) . W_2^T + b_2; y = LN_next(x)
//
// At this width a block is bound by its rows' trips through HBM: launched
// separately (LayerNorm, QKV, out-projection + LayerNorm, FFN-up, FFN-down +
// LayerNorm) each of a row's 128 columns moves 44 bytes beside attention's, most
// of them an intermediate written by one launch and read by the next.  Fused, a
// one-layer model's moves 4 + 6 (q|k|v) and 2 + 4 + 4 bytes (a layer before the last: 2 + 4 in,
// the sum 4 and h 2 out).  65536 rows, F = 128, one layer: LN + QKV 32.5 -> 19.8 us
// (4.2 TB/s), the rest 69.8 -> 25.2 us (3.3 TB/s; bound by its chain of
// hand-overs between the waves, two workgroups per CU).
//
// A workgroup of four waves takes 64 rows at a time.  As in the whole-forward
// kernel (tk_small.hip) wave w owns columns [32w, 32w + 32) of every 128-wide
// product, C^T = W . A^T on v_mfma_f32_32x32x16_f16: the residual stream stays in
// registers in the accumulator layout (lane l holds 4 consecutive columns of row
// l & 31 per 4 registers, two row blocks), activations pass between the waves
// through swizzled LDS tiles, weights are fragments packed one contiguous
// kilobyte each.  The workgroups are persistent (two per CU) and keep their
// weight fragments in registers over all their rows (F = 128; wider FFNs re-read
// W_1 and W_2 from L2 per 64 rows); the next rows' x and ctx are on their way
// while these are computed.
#include "tk_common.hpp"

namespace tk {
namespace {

constexpr int kD = 128;          // d_model = attention width
constexpr int kRows = 64;        // rows per trip
constexpr int kPitch = 2 * kD;   // bytes of an LDS tile row (128 fp16)
constexpr int kFrag = 64 * 8;    // halves per packed fragment
constexpr int kFrags = kD / 16;  // fragments of a 32-row weight block

struct NarrowArgs {
  const float* x;  // residual in
  const f16* ctx;
  const f16* w_qkv;  // packed blocks (32 rows x 128 columns): 12
  const f16* w_o;    // 4
  const f16* w_1;    // 4 per 128 FFN columns
  const f16* w_2;    // 4 per 128 FFN columns
  const float *b_qkv, *b_o, *b_1, *b_2;
  const float *n1_w, *n1_b;  // narrow_qkv: its LayerNorm; narrow_tail: LN2
  const float *n2_w, *n2_b;  // narrow_tail: the next LayerNorm
  float* sum_out;            // nullable: x after the block
  void* out;                 // q|k|v, or y
  const uint8_t* row_valid;
  float n1_eps, n2_eps;
  int T, nf, zero_all;
};

__device__ __forceinline__ int act_off(int r, int c) { return r * kPitch + ((c ^ (r & 15)) << 4); }

// LDS hand-over barrier: this wave's LDS accesses complete, global loads may stay in flight.
__device__ __forceinline__ void lds_sync() {
  __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (0 << 8) | (3 << 14));  // lgkmcnt(0)
  lds_barrier();
}

struct Lanes {
  int lane, w, g, rl;
  __device__ __forceinline__ Lanes() {
    lane = threadIdx.x & 63;
    w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    g = lane >> 5;
    rl = lane & 31;
  }
  // Through an empty asm, once per phase: the swizzled LDS addresses are then
  // formed where they are used instead of being kept in registers over all trips
  // (they spilled 50-120 B per lane).
  __device__ __forceinline__ void refresh() { asm volatile("" : "+v"(lane), "+v"(g), "+v"(rl)); }
};

__device__ __forceinline__ f16x8 wfrag(const f16* packed, int block, int kk, int lane) {
  return *reinterpret_cast<const f16x8*>(packed + ((int64_t)block * kFrags + kk) * kFrag + (uint32_t)(lane * 8));
}

// This lane's 16 columns of rows m0 + 32 i + rl (rows past T: row T - 1's).
__device__ __forceinline__ void load_rows(const float* x, int m0, int T, const Lanes& t, f32x16 (&v)[2]) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const float* r = x + (int64_t)min(m0 + 32 * i + t.rl, T - 1) * kD + 32 * t.w + 4 * t.g;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f32x4 p = *reinterpret_cast<const f32x4*>(r + 8 * q);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[i][4 * q + e] = p[e];
    }
  }
}

__device__ __forceinline__ void product(f32x16 (&acc)[2], const f16x8 (&wf)[kFrags], const char* tile, const Lanes& t,
                                        bool first) {
#pragma unroll
  for (int kk = 0; kk < kFrags; ++kk)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const f16x8 a = *reinterpret_cast<const f16x8*>(tile + act_off(32 * i + t.rl, 2 * kk + t.g));
      acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wf[kk], a, first && kk == 0 ? f32x16{} : acc[i], 0, 0, 0);
    }
}

// Mean and rstd of each row: two-pass within the wave's 32 columns, the four
// waves' (mean, M2) merged (Chan, Golub and LeVeque).  One hand-over; the caller
// separates two uses of `stats` by a barrier.
__device__ __forceinline__ void row_stats(const f32x16 (&v)[2], f32x2* stats, const Lanes& t, float eps,
                                          float (&mean)[2], float (&rstd)[2]) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    float s = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) s += v[i][r];
    const float mw = pair_sum(s) * (1.f / 32);
    s = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float d = v[i][r] - mw;
      s += d * d;
    }
    s = pair_sum(s);
    if (t.g == 0) stats[t.w * kRows + 32 * i + t.rl] = f32x2{mw, s};
  }
  lds_sync();
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int m = 32 * i + t.rl;
    const f32x2 s0 = stats[m], s1 = stats[kRows + m], s2 = stats[2 * kRows + m], s3 = stats[3 * kRows + m];
    mean[i] = (s0[0] + s1[0] + s2[0] + s3[0]) * 0.25f;
    const float d0 = s0[0] - mean[i], d1 = s1[0] - mean[i], d2 = s2[0] - mean[i], d3 = s3[0] - mean[i];
    const float m2 = (s0[1] + s1[1] + s2[1] + s3[1]) + 32.f * (d0 * d0 + d1 * d1 + d2 * d2 + d3 * d3);
    rstd[i] = 1.0f / sqrtf(m2 * (1.f / kD) + eps);
  }
}

__device__ __forceinline__ f16x4 to_half4(const float (&v)[4]) {
  return f16x4{(f16)v[0], (f16)v[1], (f16)v[2], (f16)v[3]};
}

// Normalised rows as fp16 into a tile.
__device__ __forceinline__ void norm_to_tile(const f32x16 (&v)[2], const float (&mean)[2], const float (&rstd)[2],
                                             const float* gw, const float* gb, char* tile, const Lanes& t) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int n = 32 * t.w + 8 * q + 4 * t.g;
    const f32x4 wv = *reinterpret_cast<const f32x4*>(gw + n), bv = *reinterpret_cast<const f32x4*>(gb + n);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      float y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = (v[i][4 * q + e] - mean[i]) * rstd[i] * wv[e] + bv[e];
      *reinterpret_cast<f16x4*>(tile + act_off(32 * i + t.rl, n >> 3) + (n & 7) * 2) = to_half4(y);
    }
  }
}

__global__ __launch_bounds__(256, 2) void narrow_qkv_kernel(NarrowArgs p) {
  constexpr int kOutPitch = 3 * kPitch;  // 384 fp16
  __shared__ __attribute__((aligned(16))) char smem[kRows * kPitch + kRows * kOutPitch + 4 * kRows * 8 + 5 * kD * 4];
  char* H = smem;
  char* O = smem + kRows * kPitch;
  f32x2* stats = reinterpret_cast<f32x2*>(O + kRows * kOutPitch);
  float* vec = reinterpret_cast<float*>(stats + 4 * kRows);  // n1_w, n1_b, b_qkv
  Lanes t;
  const int tid = threadIdx.x;
  if (tid < kD) {
    vec[tid] = p.n1_w[tid];
    vec[kD + tid] = p.n1_b[tid];
  }
  for (int i = tid; i < 3 * kD; i += 256) vec[2 * kD + i] = p.b_qkv[i];
  f16x8 wq[3][kFrags];
#pragma unroll
  for (int j = 0; j < 3; ++j)
#pragma unroll
    for (int kk = 0; kk < kFrags; ++kk) wq[j][kk] = wfrag(p.w_qkv, t.w + 4 * j, kk, t.lane);
  const int trips = (p.T + kRows - 1) / kRows;
  f32x16 x[2];
  load_rows(p.x, blockIdx.x * kRows, p.T, t, x);
  lds_sync();  // vectors staged
  for (int c = blockIdx.x; c < trips; c += gridDim.x) {
    const int m0 = c * kRows;
    t.refresh();
    float mean[2], rstd[2];
    row_stats(x, stats, t, p.n1_eps, mean, rstd);
    norm_to_tile(x, mean, rstd, vec, vec + kD, H, t);
    if (c + (int)gridDim.x < trips) load_rows(p.x, (c + gridDim.x) * kRows, p.T, t, x);
    lds_sync();  // h complete (and the last trip's output rows read)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      t.refresh();
      f32x16 acc[2];
      product(acc, wq[j], H, t, true);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int n = 32 * t.w + 8 * q + 4 * t.g;
        const f32x4 bv = *reinterpret_cast<const f32x4*>(vec + (2 + j) * kD + n);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = acc[i][4 * q + e] + bv[e];
          const int r = 32 * i + t.rl, ch = (n >> 3) ^ (r & 15);
          *reinterpret_cast<f16x4*>(O + r * kOutPitch + j * kPitch + (ch << 4) + (n & 7) * 2) = to_half4(v);
        }
      }
    }
    lds_sync();  // output rows complete
    f16* dst = reinterpret_cast<f16*>(p.out) + (int64_t)m0 * 3 * kD;
#pragma unroll
    for (int u = 0; u < kRows * 48 / 256; ++u) {
      const int idx = u * 256 + tid, r = idx / 48, cc = idx % 48;
      if (m0 + r < p.T)
        *reinterpret_cast<f16x8*>(dst + r * 3 * kD + cc * 8) = *reinterpret_cast<const f16x8*>(
            O + r * kOutPitch + (cc >> 4) * kPitch + (((cc & 15) ^ (r & 15)) << 4));
    }
  }
}

// FINAL: y is fp32 (else fp16).  NF1: F = 128, the FFN's fragments stay in registers.
template <bool FINAL, bool NF1>
__global__ __launch_bounds__(256, 2) void narrow_tail_kernel(NarrowArgs p) {
  __shared__ __attribute__((aligned(16))) char smem[3 * kRows * kPitch + 4 * kRows * 8 + 6 * kD * 4];
  char* C = smem;                       // ctx
  char* H = smem + kRows * kPitch;      // h, then y (fp16)
  char* U = smem + 2 * kRows * kPitch;  // gelu(h . W_1^T + b_1)
  f32x2* stats = reinterpret_cast<f32x2*>(smem + 3 * kRows * kPitch);
  float* vec = reinterpret_cast<float*>(stats + 4 * kRows);  // b_o, n1_w, n1_b, b_2, n2_w, n2_b
  Lanes t;
  const int tid = threadIdx.x;
  if (tid < kD) {
    vec[tid] = p.b_o[tid];
    vec[kD + tid] = p.n1_w[tid];
    vec[2 * kD + tid] = p.n1_b[tid];
    vec[3 * kD + tid] = p.b_2[tid];
    vec[4 * kD + tid] = p.n2_w[tid];
    vec[5 * kD + tid] = p.n2_b[tid];
  }
  // Wave w's quarter of 64 ctx rows, global -> LDS (1 KB: 4 rows; the lane fetches
  // the chunk that the tile's swizzle keeps at its place).
  const uint32_t c_lds = (uint32_t)(size_t)(lds_char*)C + t.w * 4096;
  auto fetch_ctx = [&](int m0) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int r = 16 * t.w + 4 * u + (t.lane >> 4);
      const int ch = (t.lane & 15) ^ (r & 15);
      dma16(p.ctx + (int64_t)min(m0 + r, p.T - 1) * kD + ch * 8, c_lds + u * 1024);
    }
  };
  const int trips = (p.T + kRows - 1) / kRows;
  fetch_ctx(blockIdx.x * kRows);
  f32x16 x[2], xn[2];
  load_rows(p.x, blockIdx.x * kRows, p.T, t, xn);
  f16x8 wo[kFrags], w1[kFrags], w2[kFrags];
#pragma unroll
  for (int kk = 0; kk < kFrags; ++kk) {
    wo[kk] = wfrag(p.w_o, t.w, kk, t.lane);
    if constexpr (NF1) {
      w1[kk] = wfrag(p.w_1, t.w, kk, t.lane);
      w2[kk] = wfrag(p.w_2, t.w, kk, t.lane);
    }
  }
  for (int c = blockIdx.x; c < trips; c += gridDim.x) {
    const int m0 = c * kRows, next = c + gridDim.x;
    t.refresh();
    wait_vmcnt<0>();  // this wave's ctx rows are in LDS
    lds_sync();
    f32x16 acc[2];
    product(acc, wo, C, t, true);
    bool valid[2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
      valid[i] = p.row_valid == nullptr || p.row_valid[min(m0 + 32 * i + t.rl, p.T - 1)] != 0;
    // x + ctx . W_o^T + b_o; a padded row's attention output is 0
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f32x4 bv = *reinterpret_cast<const f32x4*>(vec + 32 * t.w + 8 * q + 4 * t.g);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float r = xn[i][4 * q + e];
          x[i][4 * q + e] = valid[i] ? acc[i][4 * q + e] + (bv[e] + r) : r;
        }
    }
    t.refresh();
    float mean[2], rstd[2];
    row_stats(x, stats, t, p.n1_eps, mean, rstd);  // (its barrier: every wave is done with C)
    if (next < trips) {
      fetch_ctx(next * kRows);
      load_rows(p.x, next * kRows, p.T, t, xn);
    }
    norm_to_tile(x, mean, rstd, vec + kD, vec + 2 * kD, H, t);
    lds_sync();
    f32x16 acc2[2];
    for (int f = 0; f < (NF1 ? 1 : p.nf); ++f) {
      t.refresh();
      if constexpr (!NF1) {
#pragma unroll
        for (int kk = 0; kk < kFrags; ++kk) {
          w1[kk] = wfrag(p.w_1, 4 * f + t.w, kk, t.lane);
          w2[kk] = wfrag(p.w_2, 4 * f + t.w, kk, t.lane);
        }
        if (f > 0) lds_sync();  // the last columns' U has been read
      }
      product(acc, w1, H, t, true);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int n = 32 * t.w + 8 * q + 4 * t.g;
        const f32x4 bv = *reinterpret_cast<const f32x4*>(p.b_1 + f * kD + n);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = gelu_erf(acc[i][4 * q + e] + bv[e]);
          *reinterpret_cast<f16x4*>(U + act_off(32 * i + t.rl, n >> 3) + (n & 7) * 2) = to_half4(v);
        }
      }
      t.refresh();
      lds_sync();
      product(acc2, w2, U, t, NF1 || f == 0);
    }
    // x + u . W_2^T + b_2; a padded row's block output is 0
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f32x4 bv = *reinterpret_cast<const f32x4*>(vec + 3 * kD + 32 * t.w + 8 * q + 4 * t.g);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          x[i][4 * q + e] = valid[i] ? acc2[i][4 * q + e] + (bv[e] + x[i][4 * q + e]) : 0.f;
    }
    if (p.sum_out) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int m = m0 + 32 * i + t.rl;
        if (m < p.T) {
          float* r = p.sum_out + (int64_t)m * kD + 32 * t.w + 4 * t.g;
#pragma unroll
          for (int q = 0; q < 4; ++q)
            *reinterpret_cast<f32x4*>(r + 8 * q) =
                f32x4{x[i][4 * q], x[i][4 * q + 1], x[i][4 * q + 2], x[i][4 * q + 3]};
        }
      }
    }
    t.refresh();
    row_stats(x, stats, t, p.n2_eps, mean, rstd);
    if constexpr (FINAL) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int n = 32 * t.w + 8 * q + 4 * t.g;
        const f32x4 wv = *reinterpret_cast<const f32x4*>(vec + 4 * kD + n);
        const f32x4 bv = *reinterpret_cast<const f32x4*>(vec + 5 * kD + n);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int m = m0 + 32 * i + t.rl;
          const bool zero = !valid[i] && p.zero_all;
          f32x4 y;
#pragma unroll
          for (int e = 0; e < 4; ++e) y[e] = zero ? 0.f : (x[i][4 * q + e] - mean[i]) * rstd[i] * wv[e] + bv[e];
          if (m < p.T) *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(p.out) + (int64_t)m * kD + n) = y;
        }
      }
    } else {
      norm_to_tile(x, mean, rstd, vec + 4 * kD, vec + 5 * kD, H, t);  // (H: last read before the U barrier)
      lds_sync();
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int r = 16 * u + (tid >> 4), ch = tid & 15;
        if (m0 + r < p.T)
          *reinterpret_cast<f16x8*>(reinterpret_cast<f16*>(p.out) + (int64_t)(m0 + r) * kD + ch * 8) =
              *reinterpret_cast<const f16x8*>(H + act_off(r, ch));
      }
    }
  }
}

constexpr int kGrid = 512;  // two workgroups per CU

bool al16(const void* q) { return ((uintptr_t)q & 15) == 0; }

}  // namespace
}  // namespace tk

using namespace tk;

extern "C" int tk_narrow_supported(int64_t d_model, int64_t attn_width, int64_t ffn_dim) {
  return d_model == kD && attn_width == kD && ffn_dim >= kD && ffn_dim % kD == 0 && ffn_dim <= 1024;
}

extern "C" int tk_narrow_qkv(const float* x, const float* ln_w, const float* ln_b, float eps, const tk_half* w_packed,
                             const float* b_qkv, tk_half* qkv, int64_t rows, void* stream) {
  TK_REQUIRE(x && ln_w && ln_b && w_packed && b_qkv && qkv, TK_ERR_ARG, "tk_narrow_qkv: null pointer");
  TK_REQUIRE(rows >= 0 && rows < (1ll << 31) - kRows, TK_ERR_ARG, "tk_narrow_qkv: rows=%lld", (long long)rows);
  TK_REQUIRE(al16(x) && al16(w_packed) && al16(qkv), TK_ERR_ARG, "tk_narrow_qkv: x, w and qkv must be 16-byte aligned");
  if (rows == 0) return TK_OK;
  NarrowArgs p{};
  p.x = x;
  p.n1_w = ln_w;
  p.n1_b = ln_b;
  p.n1_eps = eps;
  p.w_qkv = reinterpret_cast<const f16*>(w_packed);
  p.b_qkv = b_qkv;
  p.out = qkv;
  p.T = (int)rows;
  const int64_t trips = (rows + kRows - 1) / kRows;
  hipLaunchKernelGGL(narrow_qkv_kernel, dim3((unsigned)(trips < kGrid ? trips : kGrid)), dim3(256), 0,
                     as_stream(stream), p);
  return check_launch("tk_narrow_qkv");
}

extern "C" int tk_narrow_tail(const tk_half* ctx, const float* resid, const tk_half* w_o, const float* b_o,
                              const float* n2_w, const float* n2_b, float n2_eps, const tk_half* w_1,
                              const float* b_1, const tk_half* w_2, const float* b_2, int64_t ffn_dim,
                              const float* next_w, const float* next_b, float next_eps, float* sum_out, void* out,
                              int out_dtype, int64_t rows, const uint8_t* row_valid, int row_mode, void* stream) {
  TK_REQUIRE(ctx && resid && w_o && b_o && n2_w && n2_b && w_1 && b_1 && w_2 && b_2 && next_w && next_b && out,
             TK_ERR_ARG, "tk_narrow_tail: null pointer");
  TK_REQUIRE(tk_narrow_supported(kD, kD, ffn_dim), TK_ERR_UNSUPPORTED,
             "tk_narrow_tail: ffn_dim=%lld must be a multiple of 128 up to 1024", (long long)ffn_dim);
  TK_REQUIRE(rows >= 0 && rows < (1ll << 31) - kRows, TK_ERR_ARG, "tk_narrow_tail: rows=%lld", (long long)rows);
  TK_REQUIRE(out_dtype == TK_F16 || out_dtype == TK_F32, TK_ERR_ARG, "tk_narrow_tail: bad out_dtype");
  TK_REQUIRE(row_valid == nullptr || row_mode == TK_ROWS_ZERO || row_mode == TK_ROWS_ZERO_ALL, TK_ERR_ARG,
             "tk_narrow_tail: bad row_mode %d", row_mode);
  // zeroed normalised rows only where the result is the final norm
  TK_REQUIRE(row_valid == nullptr || row_mode != TK_ROWS_ZERO_ALL || out_dtype == TK_F32, TK_ERR_UNSUPPORTED,
             "tk_narrow_tail: TK_ROWS_ZERO_ALL needs fp32 output");
  TK_REQUIRE(al16(ctx) && al16(resid) && al16(w_o) && al16(w_1) && al16(w_2) && al16(b_1) && al16(sum_out) && al16(out),
             TK_ERR_ARG, "tk_narrow_tail: buffers must be 16-byte aligned");
  if (rows == 0) return TK_OK;
  NarrowArgs p{};
  p.ctx = reinterpret_cast<const f16*>(ctx);
  p.x = resid;
  p.w_o = reinterpret_cast<const f16*>(w_o);
  p.w_1 = reinterpret_cast<const f16*>(w_1);
  p.w_2 = reinterpret_cast<const f16*>(w_2);
  p.b_o = b_o;
  p.b_1 = b_1;
  p.b_2 = b_2;
  p.n1_w = n2_w;
  p.n1_b = n2_b;
  p.n1_eps = n2_eps;
  p.n2_w = next_w;
  p.n2_b = next_b;
  p.n2_eps = next_eps;
  p.sum_out = sum_out;
  p.out = out;
  p.row_valid = row_valid;
  p.zero_all = row_mode == TK_ROWS_ZERO_ALL;
  p.T = (int)rows;
  p.nf = (int)(ffn_dim / kD);
  const int64_t trips = (rows + kRows - 1) / kRows;
  const dim3 grid((unsigned)(trips < kGrid ? trips : kGrid)), block(256);
  hipStream_t st = as_stream(stream);
  const bool fin = out_dtype == TK_F32, one = p.nf == 1;
  if (fin && one) hipLaunchKernelGGL((narrow_tail_kernel<true, true>), grid, block, 0, st, p);
  else if (fin) hipLaunchKernelGGL((narrow_tail_kernel<true, false>), grid, block, 0, st, p);
  else if (one) hipLaunchKernelGGL((narrow_tail_kernel<false, true>), grid, block, 0, st, p);
  else hipLaunchKernelGGL((narrow_tail_kernel<false, false>), grid, block, 0, st, p);
  return check_launch("tk_narrow_tail");
}
