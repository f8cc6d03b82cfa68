// Row kernels of the attention block at 96 and 192 channels (AttnBlock,
// packages/shrimp/python/shrimp/model.py:448-514), the widths whose weights
// either do not fit a workgroup's LDS (192: 368 KB of MLP weights) or leave a
// persistent workgroup with too few rows (96):
//   qkv:  n = LN1(seq); [q | k | v] = n Wqkv^T + bqkv, head-major
//   mlp:  s1 = seq + g_attn m (att Wo^T + bo); h = GELU(LN2(s1) W1^T + b1);
//         seq = s1 + g_mlp m (h W2^T + b2), s1 in fp32, token low parts as mlp.hip
// with the same folded, packed weights and the same product orientation and
// fragment orders as qkv.hip and mlp.hip. As exact as the linear_kernel sequence
// before them: two-pass variances and gelu_fine (3 us of the 192-channel MLP
// together, 1.5 of the 96-channel one).
//
// One workgroup: four waves, MB blocks of 16 rows each, whose activations stay
// in registers from the first load to the last store. The weights pass through
// a ring of three LDS stages (at most 24 fragments of 1 KiB each) by DMA two
// stages ahead, so every fragment is read from L2 once per 64 MB rows and feeds
// 4 MB row blocks. Requests retire in order (vmcnt): at the top of a stage its
// DMAs, issued two stages earlier, are complete once at most the requests of
// the previous stage are outstanding. LDS reads go through integer addresses
// (through a pointer the compiler waits for the DMAs in flight).
//
// They replace linear_kernel (two output blocks per pass over the rows, the
// LayerNorm redone by each of 18 column groups, the hidden rows through HBM) in
// the attention block. 192 channels, 64 824 rows: qkv 122.8 -> 31.9 us (102 MB,
// 3.2 TB/s), out_proj + fc1 + fc2 152.8 -> 53.0 us (24 GFLOP, 450 TFLOP/s). 96
// channels, 49 200 rows: qkv with the zeroed pads 41.3 -> 19.4 us, MLP 58.9 ->
// 19.4 us. Bound: latency, no unit is at its limit (a copy reaches 5.2 TB/s;
// counters at 192 channels: qkv VALU 0.18 and MFMA 0.16 of the launch's cycles, MLP
// 0.32 and 0.18): one and a half waves per SIMD over the launch, in one chain each
// of rows, stages behind a barrier, and 8-byte stores.
#include <algorithm>

#include "capi.hpp"
#include "common.hpp"

namespace shrimp {

__global__ void pack_weight_kernel(const float* __restrict__ src, unsigned short* __restrict__ dst,
                                   int K, int NOUT, int cin, int cin_pad, int64_t s_t,
                                   int64_t s_c, int64_t s_n, int interleaved);
__global__ void scale_rows_cols_kernel(const float* __restrict__ src, const float* __restrict__ rs,
                                       const float* __restrict__ cs, int n_out, int n_in,
                                       float* __restrict__ dst);

namespace {

typedef __attribute__((address_space(3))) void lds_dst_t;

constexpr int BW = 4;       // waves per workgroup
constexpr int STAGE = 24;   // fragments per ring slot

SHRIMP_DEV int lds_base(const void* p) {
  return (int)(uintptr_t)(__attribute__((address_space(3))) const unsigned char*)p;
}
SHRIMP_DEV u32x4 lds_frag(int addr) {
  return *(__attribute__((address_space(3))) const u32x4*)(uintptr_t)(unsigned)addr;
}
SHRIMP_DEV f32x4 lds_f4(int addr) {
  return *(__attribute__((address_space(3))) const f32x4*)(uintptr_t)(unsigned)addr;
}

// s_waitcnt vmcnt(N) alone (expcnt and lgkmcnt at their maxima)
template <int N>
SHRIMP_DEV void wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

// ---- packed weights: byte offsets -------------------------------------------------
constexpr uint32_t qkv_bias_off(int C) { return (uint32_t)(3 * C * C * 2); }
constexpr uint32_t qkv_pack_bytes(int C) { return qkv_bias_off(C) + 3 * C * 4; }
// [Wo | W1 | W2 | bo' (C) | b1' (2C) | b2' (C)]
constexpr uint32_t mlp_w1_off(int C) { return (uint32_t)(C * C * 2); }
constexpr uint32_t mlp_w2_off(int C) { return (uint32_t)(3 * C * C * 2); }
constexpr uint32_t mlp_bias_off(int C) { return (uint32_t)(5 * C * C * 2); }
constexpr uint32_t mlp_pack_bytes(int C) { return mlp_bias_off(C) + 4 * C * 4; }

constexpr uint32_t ring_bytes() { return 3 * STAGE * 1024; }

// ---- LN1 + q/k/v ---------------------------------------------------------------------
// Stage: OB blocks of 16 outputs over all KS channel chunks.
template <int C, int MB>
__global__ __launch_bounds__(BW * 64, 2) void qkv_stream_kernel(const shrimp_qkv_args a,
                                                                uint32_t x_bytes, uint32_t q_bytes,
                                                                int inv_d) {
  constexpr int KS = C / 32, NB = 3 * C / 16, OB = C == 96 ? 6 : 4;
  constexpr int NST = NB / OB, SF = OB * KS, DPW = SF / BW;
  constexpr int WAIT = DPW + OB * MB;  // fewest requests of a wave per stage
  static_assert(NB % OB == 0 && SF <= STAGE, "whole stages");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int lane = threadIdx.x & 63, wave = wave_id();
  const int lr = lane & 15, lg = lane >> 4;
  const int lds0 = lds_base(smem), bias0 = lds0 + (int)ring_bytes();
  const __amdgpu_buffer_rsrc_t wr = make_rsrc(a.packed, qkv_bias_off(C));
  const __amdgpu_buffer_rsrc_t xr = make_rsrc(a.x, x_bytes);
  const __amdgpu_buffer_rsrc_t qr = make_rsrc(a.qkv, q_bytes);
  // fragment f of stage g: chunk f / OB, output block g OB + f % OB
  auto dma = [&](int g, int slot) {
#pragma unroll
    for (int i = 0; i < (SF + BW - 1) / BW; ++i) {
      const int f = wave + BW * i;
      const int ks = f / OB, nb = g * OB + (f - ks * OB);
      if (SF % BW == 0 || f < SF)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            wr, (lds_dst_t*)(smem + (slot * STAGE + f) * 1024), 16,
            g < NST ? (uint32_t)((ks * NB + nb) * 1024 + lane * 16) : SHRIMP_OOB_OFFSET, 0, 0, 0);
    }
  };
  dma(0, 0);
  dma(1, 1);
  {
    const float* pb = reinterpret_cast<const float*>(static_cast<const unsigned char*>(a.packed) +
                                                     qkv_bias_off(C));
    float* bl = reinterpret_cast<float*>(smem + ring_bytes());
    for (int i = threadIdx.x; i < 3 * C; i += BW * 64) bl[i] = pb[i];
  }
  const int row0 = (int)blockIdx.x * (BW * 16 * MB) + wave * 16 * MB;
  u32x4 hf[MB][KS];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int row = row0 + mb * 16 + lr;
    const uint32_t xo =
        row < a.rows ? (uint32_t)((int64_t)row * a.x_sr * 2) + (uint32_t)(lg * 16) : SHRIMP_OOB_OFFSET;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) hf[mb][ks] = buf_load16(xr, xo + ks * 64);
  }
  // LayerNorm without affine (folded into the weights); absent rows give zeros
  int64_t rowbase[MB];
  bool rv[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int row = row0 + mb * 16 + lr;
    rv[mb] = row < a.rows;
    const int bq = rv[mb] ? row / a.S : 0, sq = rv[mb] ? row - bq * a.S : 0;
    rowbase[mb] = ((int64_t)bq * a.H * a.S + sq) * a.dpad;
    float s = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int w = 0; w < 4; ++w) s += bf16_lo(hf[mb][ks][w]) + bf16_hi(hf[mb][ks][w]);
    const float mean = sum_groups_swap(s) * (1.0f / C);
    float q = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const float u0 = bf16_lo(hf[mb][ks][w]) - mean, u1 = bf16_hi(hf[mb][ks][w]) - mean;
        q = fmaf(u0, u0, fmaf(u1, u1, q));
      }
    const float rstd = rsqrtf(sum_groups_swap(q) * (1.0f / C) + a.eps);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int w = 0; w < 4; ++w)
        hf[mb][ks][w] = pack_bf16x2((bf16_lo(hf[mb][ks][w]) - mean) * rstd,
                                    (bf16_hi(hf[mb][ks][w]) - mean) * rstd);
  }
  const int d = C / a.H;
  const int64_t plane = (int64_t)a.B * a.H * a.S * a.dpad, hstride = (int64_t)a.S * a.dpad;
  // the four channels c .. c + 3 (of 3 C) of row block mb; absent rows past the
  // resource (dropped), so every wave issues the same requests per stage
  auto put = [&](int mb, int nb, u32x2 pk) {
    const int which = nb / (C / 16);
    const int within = (nb - which * (C / 16)) * 16 + lg * 4;
    const int head = (within * inv_d) >> 16;
    const int dd = within - head * d;
    const uint32_t off = rv[mb] ? (uint32_t)((rowbase[mb] + which * plane + head * hstride + dd) * 2)
                                : SHRIMP_OOB_OFFSET;
    __builtin_amdgcn_raw_buffer_store_b64(pk, qr, off, 0, 0);
  };
  int slot = 0;
#pragma unroll 1
  for (int g = 0; g < NST; ++g) {
    __builtin_amdgcn_sched_barrier(0);
    if (g == 0) wait_vm<0>();
    else wait_vm<WAIT>();
    __syncthreads();
    dma(g + 2, slot == 0 ? 2 : slot - 1);
    __builtin_amdgcn_sched_barrier(0);
    const int wbase = lds0 + slot * STAGE * 1024 + lane * 16;
#pragma unroll
    for (int o = 0; o < OB; ++o) {
      const int nb = g * OB + o;
      const f32x4 bb = lds_f4(bias0 + (nb * 16 + lg * 4) * 4);
      f32x4 acc[MB];
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) acc[mb] = bb;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const u32x4 w = lds_frag(wbase + (ks * OB + o) * 1024);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[mb] = mfma16x16x32(w, hf[mb][ks], acc[mb]);
      }
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
        put(mb, nb, u32x2{pack_bf16x2(acc[mb][0], acc[mb][1]), pack_bf16x2(acc[mb][2], acc[mb][3])});
    }
    slot = slot == 2 ? 0 : slot + 1;
  }
  // zero columns d .. dpad - 1 of every head (the attention's padded channels)
  const int pad4 = (a.dpad - d) / 4;
  for (int i = lane; i < 3 * a.H * pad4 * 16 * MB; i += 64) {
    const int r = i / (3 * a.H * pad4), k = i - r * (3 * a.H * pad4);
    const int hw = k / pad4, e = d + (k - hw * pad4) * 4;
    const int row = row0 + r;
    const int bq = row / a.S, sq = row - bq * a.S;
    const int which = hw / a.H, head = hw - which * a.H;
    const uint32_t off =
        row < a.rows ? (uint32_t)((((int64_t)bq * a.H * a.S + sq) * a.dpad + which * plane +
                                   head * hstride + e) * 2)
                     : SHRIMP_OOB_OFFSET;
    __builtin_amdgcn_raw_buffer_store_b64(u32x2{0u, 0u}, qr, off, 0, 0);
  }
}

// ---- out_proj + residual + LN2 + fc1 + GELU + fc2 + residual --------------------------
// Stages: out_proj, OB output blocks each; then HB 32-wide hidden slices each
// (the slice's fc1 fragments, then its fc2 fragments).
template <int C, int MB>
__global__ __launch_bounds__(BW * 64, 2) void mlp_stream_kernel(const shrimp_mlp_args a,
                                                                uint32_t x_bytes, uint32_t s_bytes,
                                                                uint32_t lo_bytes) {
  constexpr int KS = C / 32, NB = C / 16, NBH = 2 * NB, KT = 2 * KS;
  constexpr int OB = STAGE / KS < NB ? STAGE / KS : NB, NSO = NB / OB, SFO = OB * KS;
  constexpr int SLF = 2 * KS + NB, HB = STAGE / SLF, NSH = KT / HB, SFH = HB * SLF;
  constexpr int NST = NSO + NSH;
  constexpr int DPW = (SFO < SFH ? SFO : SFH) / BW;  // fewest DMAs of a wave per stage
  static_assert(NB % OB == 0 && KT % HB == 0 && SFO <= STAGE && SFH <= STAGE, "whole stages");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int lane = threadIdx.x & 63, wave = wave_id();
  const int lr = lane & 15, lg = lane >> 4;
  const int lds0 = lds_base(smem), bias0 = lds0 + (int)ring_bytes();
  const __amdgpu_buffer_rsrc_t wr = make_rsrc(a.packed, mlp_bias_off(C));
  auto dma = [&](int g, int slot) {
#pragma unroll
    for (int i = 0; i < STAGE / BW; ++i) {
      const int f = wave + BW * i;
      uint32_t off = SHRIMP_OOB_OFFSET;
      bool on = true;
      if (g < NSO) {
        on = f < SFO;
        const int ks = f / OB, nb = g * OB + (f - ks * OB);
        off = (uint32_t)((ks * NB + nb) * 1024);
      } else if (g < NST) {
        on = f < SFH;
        const int sl = f / SLF, r = f - sl * SLF, kt = (g - NSO) * HB + sl;
        // fc1: chunk r / 2, hidden block 2 kt + r % 2; fc2: chunk kt, output block
        off = r < 2 * KS ? mlp_w1_off(C) + (uint32_t)(((r >> 1) * NBH + 2 * kt + (r & 1)) * 1024)
                         : mlp_w2_off(C) + (uint32_t)((kt * NB + (r - 2 * KS)) * 1024);
      } else {
        on = f < SFH;
      }
      if (on)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            wr, (lds_dst_t*)(smem + (slot * STAGE + f) * 1024), 16,
            off == SHRIMP_OOB_OFFSET ? off : off + (uint32_t)(lane * 16), 0, 0, 0);
    }
  };
  dma(0, 0);
  dma(1, 1);
  {
    const float* pb = reinterpret_cast<const float*>(static_cast<const unsigned char*>(a.packed) +
                                                     mlp_bias_off(C));
    float* bl = reinterpret_cast<float*>(smem + ring_bytes());
    for (int i = threadIdx.x; i < 4 * C; i += BW * 64) bl[i] = pb[i];
  }
  const __amdgpu_buffer_rsrc_t xr = make_rsrc(a.x, x_bytes);
  const __amdgpu_buffer_rsrc_t sr = make_rsrc(a.seq, s_bytes);
  const __amdgpu_buffer_rsrc_t lor = make_rsrc(a.tok_lo, lo_bytes);
  const __amdgpu_buffer_rsrc_t mr = make_rsrc(a.mask, (uint32_t)a.rows);
  const int row0 = (int)blockIdx.x * (BW * 16 * MB) + wave * 16 * MB;
  u32x4 hf[MB][KS];
  uint32_t so[MB], lo[MB];  // this lane's byte offsets in seq and in the token low parts
  unsigned live[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int row = row0 + mb * 16 + lr;
    const bool rv = row < a.rows;
    const int pos = rv ? row / a.S : 0, srow = rv ? row - pos * a.S : a.S;
    live[mb] = (unsigned)__builtin_amdgcn_raw_buffer_load_b8(
        mr, rv ? (uint32_t)row : SHRIMP_OOB_OFFSET, 0, 0);
    so[mb] = rv ? (uint32_t)((int64_t)row * a.s_sr * 2) + (uint32_t)(lg * 8) : SHRIMP_OOB_OFFSET;
    lo[mb] = srow < a.n_tokens ? (uint32_t)(((pos * a.n_tokens + srow) * C + lg * 4) * 2)
                               : SHRIMP_OOB_OFFSET;
    const uint32_t xo =
        rv ? (uint32_t)((int64_t)row * a.x_sr * 2) + (uint32_t)(lg * 16) : SHRIMP_OOB_OFFSET;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) hf[mb][ks] = buf_load16(xr, xo + ks * 64);
  }
  // the out_proj accumulators start from the residual rows and their low parts
  // (zeros for cells); bo' follows with the stage barrier, when it is in LDS
  f32x4 acc[MB][NB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const u32x2 s = buf_load8(sr, so[mb] + nb * 32), l = buf_load8(lor, lo[mb] + nb * 32);
      acc[mb][nb] = f32x4{bf16_lo(s.x) + bf16_lo(l.x), bf16_hi(s.x) + bf16_hi(l.x),
                          bf16_lo(s.y) + bf16_lo(l.y), bf16_hi(s.y) + bf16_hi(l.y)};
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  auto bias = [&](int n) { return lds_f4(bias0 + (n + lg * 4) * 4); };
  int slot = 0;
  auto next_stage = [&](int g) -> int {
    __builtin_amdgcn_sched_barrier(0);
    if (g == 0) wait_vm<0>();
    else wait_vm<DPW>();
    __syncthreads();
    dma(g + 2, slot == 0 ? 2 : slot - 1);
    __builtin_amdgcn_sched_barrier(0);
    const int wbase = lds0 + slot * STAGE * 1024 + lane * 16;
    slot = slot == 2 ? 0 : slot + 1;
    return wbase;
  };
#pragma unroll
  for (int g = 0; g < NSO; ++g) {
    const int wbase = next_stage(g);
#pragma unroll
    for (int o = 0; o < OB; ++o) {
      const int nb = g * OB + o;
      const f32x4 bb = bias(nb * 16);
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) acc[mb][nb] = acc[mb][nb] + bb;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const u32x4 w = lds_frag(wbase + (ks * OB + o) * 1024);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[mb][nb] = mfma16x16x32(w, hf[mb][ks], acc[mb][nb]);
      }
    }
  }
  // LayerNorm 2 (affine folded into W1', b1'); then the accumulators, s1, go on
  // as the fc2 accumulators' start
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    // two passes over the registers: E[x^2] - mean^2 cancels for rows whose mean is
    // large against their spread
    f32x4 sj = acc[mb][0];
#pragma unroll
    for (int nb = 1; nb < NB; ++nb) sj = sj + acc[mb][nb];
    const float mean = sum_groups_swap((sj[0] + sj[1]) + (sj[2] + sj[3])) * (1.0f / C);
    float qj[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float u = acc[mb][nb][j] - mean;
        qj[j] = fmaf(u, u, qj[j]);
      }
    const float rstd =
        rsqrtf(sum_groups_swap((qj[0] + qj[1]) + (qj[2] + qj[3])) * (1.0f / C) + a.eps);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const f32x4 v0 = (acc[mb][2 * ks] - mean) * rstd, v1 = (acc[mb][2 * ks + 1] - mean) * rstd;
      hf[mb][ks] = u32x4{pack_bf16x2(v0[0], v0[1]), pack_bf16x2(v0[2], v0[3]),
                         pack_bf16x2(v1[0], v1[1]), pack_bf16x2(v1[2], v1[3])};
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = acc[mb][nb] + bias(3 * C + nb * 16);
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll 1
  for (int g = NSO; g < NST; ++g) {
    const int wbase = next_stage(g);
#pragma unroll
    for (int sl = 0; sl < HB; ++sl) {
      const int kt = (g - NSO) * HB + sl;
      const int w1 = wbase + sl * SLF * 1024, w2 = w1 + 2 * KS * 1024;
      f32x4 ah[MB][2];
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        const f32x4 bb = bias(C + (2 * kt + hh) * 16);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) ah[mb][hh] = bb;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const u32x4 w = lds_frag(w1 + (2 * ks + hh) * 1024);
#pragma unroll
          for (int mb = 0; mb < MB; ++mb) ah[mb][hh] = mfma16x16x32(w, hf[mb][ks], ah[mb][hh]);
        }
      }
      u32x4 gf[MB];
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
        gf[mb] = u32x4{pack_bf16x2(gelu_fine(ah[mb][0][0]), gelu_fine(ah[mb][0][1])),
                       pack_bf16x2(gelu_fine(ah[mb][0][2]), gelu_fine(ah[mb][0][3])),
                       pack_bf16x2(gelu_fine(ah[mb][1][0]), gelu_fine(ah[mb][1][1])),
                       pack_bf16x2(gelu_fine(ah[mb][1][2]), gelu_fine(ah[mb][1][3]))};
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const u32x4 w = lds_frag(w2 + nb * 1024);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[mb][nb] = mfma16x16x32(w, gf[mb], acc[mb][nb]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // rows with mask 0 keep their residual
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const uint32_t sm = live[mb] ? so[mb] : SHRIMP_OOB_OFFSET;
    const uint32_t lm = live[mb] ? lo[mb] : SHRIMP_OOB_OFFSET;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const f32x4 v = acc[mb][nb];
      const u32x2 pk{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
      __builtin_amdgcn_raw_buffer_store_b64(pk, sr, sm + nb * 32, 0, 0);
      __builtin_amdgcn_raw_buffer_store_b64(
          u32x2{pack_bf16x2(v[0] - bf16_lo(pk.x), v[1] - bf16_hi(pk.x)),
                pack_bf16x2(v[2] - bf16_lo(pk.y), v[3] - bf16_hi(pk.y))},
          lor, lm + nb * 32, 0, 0);
    }
  }
}

// ---- packing -------------------------------------------------------------------------------

// out[n] = scale * b[n] (+ sum_k W[n][k] ln_b[k])
__global__ void fold_bias_kernel(const float* __restrict__ w, const float* __restrict__ b,
                                 const float* __restrict__ ln_b, const float* __restrict__ scale,
                                 int n_out, int n_in, float* __restrict__ out) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= n_out) return;
  float s = scale ? scale[n] * b[n] : b[n];
  if (ln_b)
    for (int k = 0; k < n_in; ++k) s = fmaf(w[(int64_t)n * n_in + k], ln_b[k], s);
  out[n] = s;
}

// dst fragments of diag(rs) W diag(cs), W (n_out, n_in), through `tmp`
void pack_scaled(const float* w, const float* rs, const float* cs, int n_out, int n_in, float* tmp,
                 unsigned char* dst, int interleaved, hipStream_t st) {
  const int64_t n = (int64_t)n_out * n_in;
  hipLaunchKernelGGL(scale_rows_cols_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, w,
                     rs, cs, n_out, n_in, tmp);
  const int64_t frags = n / 8;
  hipLaunchKernelGGL(pack_weight_kernel, dim3((unsigned)((frags + 255) / 256)), dim3(256), 0, st, tmp,
                     reinterpret_cast<unsigned short*>(dst), n_in, n_out, n_in, n_in, (int64_t)0,
                     (int64_t)1, (int64_t)n_in, interleaved);
}

}  // namespace

bool block_stream_width(int C) { return C == 96 || C == 192; }
size_t qkv_stream_pack_bytes(int C) { return qkv_pack_bytes(C); }
size_t mlp_stream_pack_bytes(int C) { return mlp_pack_bytes(C); }

int pack_qkv_stream(const float* w, const float* b, const float* ln_w, const float* ln_b,
                    unsigned char* pk, float* tmp, int C, hipStream_t st) {
  pack_scaled(w, nullptr, ln_w, 3 * C, C, tmp, pk, 0, st);
  hipLaunchKernelGGL(fold_bias_kernel, dim3((3 * C + 255) / 256), dim3(256), 0, st, w, b, ln_b,
                     (const float*)nullptr, 3 * C, C, reinterpret_cast<float*>(pk + qkv_bias_off(C)));
  return check_launch("pack_attn_qkv");
}

int pack_mlp_stream(const shrimp_mlp_weights* w, unsigned char* pk, float* tmp, hipStream_t st) {
  const int C = w->C;
  pack_scaled(w->out_w, w->g_attn, nullptr, C, C, tmp, pk, 0, st);
  pack_scaled(w->fc1_w, nullptr, w->ln_w, 2 * C, C, tmp, pk + mlp_w1_off(C), 1, st);
  pack_scaled(w->fc2_w, w->g_mlp, nullptr, C, 2 * C, tmp, pk + mlp_w2_off(C), 1, st);
  float* bo = reinterpret_cast<float*>(pk + mlp_bias_off(C));
  const dim3 t(256);
  hipLaunchKernelGGL(fold_bias_kernel, dim3((C + 255) / 256), t, 0, st, w->out_w, w->out_b,
                     (const float*)nullptr, w->g_attn, C, C, bo);
  hipLaunchKernelGGL(fold_bias_kernel, dim3((2 * C + 255) / 256), t, 0, st, w->fc1_w, w->fc1_b, w->ln_b,
                     (const float*)nullptr, 2 * C, C, bo + C);
  hipLaunchKernelGGL(fold_bias_kernel, dim3((C + 255) / 256), t, 0, st, w->fc2_w, w->fc2_b,
                     (const float*)nullptr, w->g_mlp, C, 2 * C, bo + 3 * C);
  return check_launch("pack_attn_mlp");
}

// Two row blocks per wave once that gives every compute unit a workgroup (each
// fragment read from LDS then feeds two products), else one.
static int row_blocks(int rows) { return rows >= 128 * cu_count() ? 2 : 1; }

int launch_qkv_stream(const shrimp_qkv_args* a, uint32_t x_bytes, uint32_t q_bytes, hipStream_t st) {
  const int mb = row_blocks(a->rows), per = BW * 16 * mb;
  const dim3 grid((unsigned)((a->rows + per - 1) / per)), block(BW * 64);
  const int d = a->C / a->H;
  const int inv_d = (65536 + d - 1) / d;  // floor(c / d) = c inv_d >> 16 for c < 192
  const size_t lds = ring_bytes() + 3 * a->C * 4;
#define BS_LAUNCH(CV, MBV)                                                                       \
  hipLaunchKernelGGL((qkv_stream_kernel<CV, MBV>), grid, block, lds, st, *a, x_bytes, q_bytes, inv_d)
  if (a->C == 96) {
    if (mb == 2) BS_LAUNCH(96, 2);
    else BS_LAUNCH(96, 1);
  } else {
    if (mb == 2) BS_LAUNCH(192, 2);
    else BS_LAUNCH(192, 1);
  }
#undef BS_LAUNCH
  return check_launch("attn_qkv");
}

int launch_mlp_stream(const shrimp_mlp_args* a, uint32_t x_bytes, uint32_t s_bytes, uint32_t lo_bytes,
                      hipStream_t st) {
  const int mb = row_blocks(a->rows), per = BW * 16 * mb;
  const dim3 grid((unsigned)((a->rows + per - 1) / per)), block(BW * 64);
  const size_t lds = ring_bytes() + 4 * a->C * 4;
#define BS_LAUNCH(CV, MBV)                                                                       \
  hipLaunchKernelGGL((mlp_stream_kernel<CV, MBV>), grid, block, lds, st, *a, x_bytes, s_bytes, lo_bytes)
  if (a->C == 96) {
    if (mb == 2) BS_LAUNCH(96, 2);
    else BS_LAUNCH(96, 1);
  } else {
    if (mb == 2) BS_LAUNCH(192, 2);
    else BS_LAUNCH(192, 1);
  }
#undef BS_LAUNCH
  return check_launch("attn_mlp");
}

}  // namespace shrimp
