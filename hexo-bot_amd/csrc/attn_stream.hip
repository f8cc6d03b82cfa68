// Attention with keys streamed through LDS, for head dims padded to 32 or 64
// (the 96- and 192-channel networks and the operator ABI's larger heads) at
// any sequence length. Same semantics as attn.hip: softmax(q k^T / sqrt(d) +
// bias) v, keys past seq_lens never visited, masked cells weight 0
// (packages/shrimp/python/shrimp/model.py:448-492, _triton_attn.py:59-130).
//
// One workgroup = one (position, head) and 64 QB queries (QB blocks of 16 per
// wave, four waves). K and V rows arrive 64 keys at a time by buffer-to-LDS
// DMA, two buffers, the next chunk requested under the current one's products,
// so LDS does not grow with the sequence beyond 9 bytes per key and three
// workgroups share a compute unit at D = 64 (the whole-sequence kernel held
// one, and at S > 560 did not fit at all). Rows lie as in memory (2 D bytes),
// their 16-byte pieces XOR-swizzled by row so the reads spread over the banks:
//   K: lane (lr, lg) reads piece 4 ks + lg of key lr = the A operand of a
//      16x16x32 product, two products per 16 keys x 16 queries at D = 64;
//   V: ds_read_b64_tr_b16 transposes on the way out: lanes 16 lg .. + 15 address
//      keys 4 lg .. + 3 (four lanes, 16 dims each) and lane lr receives dim lr
//      of those four keys, the A operand of V^T P^T.
// All products stay transposed (S^T = K Q^T, O^T = V^T P^T), so a lane's scores
// are already its slice of the next product's B operand.
//
// Softmax in base 2 around a per-query offset m, the largest score so far: the
// accumulators start at -m / scale, so fma(s, scale, bias) is score - m and a step
// without a new maximum has no rescale and no lane exchange. Row sums come from a
// product with ones. The largest weight is exactly 1 and so has no rounding to
// bf16: letting scores pass m by up to 2^8 saved the rescales (a tenth of a pair
// call at 60 positions) but put the error against float64 at 2.2e-3 instead of
// 2.07e-3 (bf16 operands; the whole-sequence kernel: 2.07e-3). FINE: a weight is
// two bf16 numbers, its high and low part, and multiplies V as two products.
//
// Biases, fp32 tables in LDS. LINEAR: the offsets the live cells span, laid out
// (2 dq_max + 1) x (2 dr_max + 1) without clamping while they fit MAX_OFFSETS
// (spans of 28 x 28), so a score's bias is one read at kkey[key] - qkey[query];
// CLAMP: the clamped table of wider positions (13.7 VALU per score against
// 4.8); PAIR: table rows from the pair tensor. Key blocks that hold token or
// dead keys, and waves whose queries hold tokens, select per lane.
//
// Bound: no single unit. Counters, 111 positions, S = 584, H = 3, D = 64, FINE: VALU
// issue 0.50 of the launch's cycles, MFMA 0.18, LDS 0.20; 150 positions, S = 328,
// H = 4, D = 32 0.45, 0.07 and 0.21: the VALU of a score (an address, an fma, an exp,
// half a maximum and half a pack) with two to three waves per SIMD that wait 0.4 to
// 0.5 of their time, in the chain of one chunk. Measured on MI355X: the first
// shape 1873 us (one query row per thread) -> 106 us (94 with one bf16 per weight),
// the second 67 -> 47 us; the pair tensor at 60 positions, S = 341, H = 3, D = 64
// 94 -> 25 us. Two 32-key steps per chunk as a rolled loop keep 147 VGPRs (unrolled
// 168 with 49 spilled). A query's bits depend on its own rows only, not on the tiling
// or on the queries beside it.
#include <type_traits>

#include "capi.hpp"
#include "common.hpp"

namespace shrimp {

#define AST_LOG2E 1.4426950408889634f
#define AST_NEG_BIG (-1.0e30f)

namespace {

enum : int { KEY_CELL = 0, KEY_TOKEN = 1, KEY_DEAD = 2 };
enum : int { PATH_CLAMP = 0, PATH_LINEAR = 1, PATH_PAIR = 2 };

constexpr int KC = 64;              // keys per chunk
constexpr int MAX_OFFSETS = 57 * 57;
constexpr int TU = 16;              // table rows a wave loads together
constexpr int MAX_LUT_M = 28;       // (2 M + 1)^2 entries fit the same region
// Below this an offset's rounding (2^-24 of it) is 1.5e-5 of a weight. Scoring
// again leaves a few 2^-24 of the old offset in the new one, so offsets of up to
// 1e29 settle within six times.
constexpr float FAR_OFFSET = 256.f;
constexpr int MAX_RESCORES = 8;

typedef __attribute__((address_space(3))) void lds_dst_t;
typedef __attribute__((address_space(3))) const unsigned char lds_cu8;

SHRIMP_DEV int clampi(int x, int m) { return min(max(x, -m), m); }

// LDS byte addresses as plain integers: no base pointer added per read, and
// the compiler, which takes a read through a pointer into the workgroup's LDS
// to alias the chunk DMA in flight and waits for it (vmcnt 0), leaves the
// ordering to the wait and barrier that end each chunk (2 % at D = 64, S = 584, 3 %
// for a dozen positions at D = 32).
SHRIMP_DEV int lds_addr(const void* p) { return (int)(uintptr_t)(lds_cu8*)p; }
SHRIMP_DEV unsigned lds_u32(int addr) {
  return *(__attribute__((address_space(3))) const unsigned*)(uintptr_t)(unsigned)addr;
}
SHRIMP_DEV unsigned lds_u8(int addr) {
  return *(__attribute__((address_space(3))) const unsigned char*)(uintptr_t)(unsigned)addr;
}
SHRIMP_DEV float lds_f32(int addr) {
  return *(__attribute__((address_space(3))) const float*)(uintptr_t)(unsigned)addr;
}
SHRIMP_DEV u32x4 lds_16(int addr) {
  return *(__attribute__((address_space(3))) const u32x4*)(uintptr_t)(unsigned)addr;
}
// V^T fragments of 32 keys: for each address a pair of transposing reads, RB16
// bytes (16 keys) apart. In assembly with its own wait: the builtin is taken to
// alias the next chunk's DMA, and the compiler waits for that before the first
// read of every chunk.
template <int RB16>
SHRIMP_DEV void lds_tr(const int (&at)[4], u32x2 (&a)[4], u32x2 (&b)[4]) {
  asm volatile(
      "ds_read_b64_tr_b16 %0, %8\n\tds_read_b64_tr_b16 %4, %8 offset:%12\n\t"
      "ds_read_b64_tr_b16 %1, %9\n\tds_read_b64_tr_b16 %5, %9 offset:%12\n\t"
      "ds_read_b64_tr_b16 %2, %10\n\tds_read_b64_tr_b16 %6, %10 offset:%12\n\t"
      "ds_read_b64_tr_b16 %3, %11\n\tds_read_b64_tr_b16 %7, %11 offset:%12\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(a[0]), "=&v"(a[1]), "=&v"(a[2]), "=&v"(a[3]), "=&v"(b[0]), "=&v"(b[1]), "=&v"(b[2]),
        "=&v"(b[3])
      : "v"(at[0]), "v"(at[1]), "v"(at[2]), "v"(at[3]), "n"(RB16)
      : "memory");
}
template <int RB16>
SHRIMP_DEV void lds_tr(const int (&at)[2], u32x2 (&a)[2], u32x2 (&b)[2]) {
  asm volatile(
      "ds_read_b64_tr_b16 %0, %4\n\tds_read_b64_tr_b16 %2, %4 offset:%6\n\t"
      "ds_read_b64_tr_b16 %1, %5\n\tds_read_b64_tr_b16 %3, %5 offset:%6\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(a[0]), "=&v"(a[1]), "=&v"(b[0]), "=&v"(b[1])
      : "v"(at[0]), "v"(at[1]), "n"(RB16)
      : "memory");
}

// Swizzle of row r's 16-byte pieces (D / 8 per row): a 128-byte line of LDS
// holds one row at D = 64 and two at D = 32.
template <int D>
SHRIMP_DEV int swz(int r) {
  return D == 64 ? (r & 7) : ((r >> 1) & 3);
}

// Per-wave state of its QB query blocks.
template <int D, int QB>
struct StreamQuery {
  u32x4 qf[QB][D / 32];
  f32x4 o[QB][D / 16];
  f32x4 l[QB], cinit[QB];  // row sums and -m / scale, four equal elements each
  float m[QB];
  int qkey[QB];         // LINEAR: offset code of the query
  int qq[QB], qr[QB];   // CLAMP: its coordinates
  bool qtok[QB];
};

struct StreamLds {      // LDS byte addresses
  int keys;             // LINEAR: per key the address of its table row for offset code 0;
                        // CLAMP: its coordinates
  int kcls;             // key classes, one byte each
  int tab;              // CLAMP and PAIR tables
  float tokb[3];          // (cell query, token key), (token query, cell key), (token, token)
  float inv_scale;
  int npos;
};

// Key blocks scored together, around one offset: the same at both tilings of the
// coords form, so that a query's bits do not depend on the tiling and with it on the
// batch. Two, which fit the registers of three waves per SIMD at QB = 2 (the 16-query
// tiling alone would take four: one position at S = 500, D = 32 13.2 against 15.1 us);
// four for the pair form, which has one tiling.
template <int PATH>
constexpr int stream_nkb() {
  return PATH == PATH_PAIR ? 4 : 2;
}

// NKB blocks of 16 keys from key k0, K and V rows at LDS bytes kbuf, vbuf;
// bit kb of `special` (wave-uniform): block kb selects its biases per lane.
template <int D, int QB, int PATH, bool FINE>
SHRIMP_DEV void stream_chunk(const shrimp_attn_args& a, StreamQuery<D, QB>& w, const StreamLds& s,
                             int k0, int L, int special, int kbuf, int vbuf, int lr, int lg,
                             float scale, const unsigned (&pd)[QB][stream_nkb<PATH>()]) {
  constexpr int NKB = stream_nkb<PATH>();
  constexpr int KS = D / 32, KD = D / 16, RB = 2 * D;
  f32x4 v[QB][NKB];
  const int ksw = swz<D>(lr);
  // scores against the offsets
  auto score = [&]() {
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const u32x4 kf = lds_16(kbuf + (kb * 16 + lr) * RB + (((ks * 4 + lg) ^ ksw) << 4));
#pragma unroll
        for (int qb = 0; qb < QB; ++qb)
          v[qb][kb] = mfma16x16x32(kf, w.qf[qb][ks], ks == 0 ? w.cinit[qb] : v[qb][kb]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb) {
      const int key0 = k0 + kb * 16 + lg * 4;
      u32x4 kk{0, 0, 0, 0}, kr{0, 0, 0, 0};
      if constexpr (PATH == PATH_LINEAR) {
        kk = lds_16(s.keys + key0 * 4);
      } else if constexpr (PATH == PATH_CLAMP) {
        const u32x4 a0 = lds_16(s.keys + key0 * 8), a1 = lds_16(s.keys + key0 * 8 + 16);
        kk = u32x4{a0[0], a0[2], a1[0], a1[2]};
        kr = u32x4{a0[1], a0[3], a1[1], a1[3]};
      }
      const int kv[4] = {(int)kk[0], (int)kk[1], (int)kk[2], (int)kk[3]};
      const int rv[4] = {(int)kr[0], (int)kr[1], (int)kr[2], (int)kr[3]};
      float bias[QB][4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) {
          if constexpr (PATH == PATH_LINEAR) {
            bias[qb][j] = lds_f32(kv[j] - w.qkey[qb]);
          } else if constexpr (PATH == PATH_CLAMP) {
            const int M = a.lut_m, W = 2 * M + 1;
            bias[qb][j] = lds_f32(
                s.tab + ((clampi(kv[j] - w.qq[qb], M) + M) * W + clampi(rv[j] - w.qr[qb], M) + M) * 4);
          } else {
            const int p = (int)((pd[qb][kb] >> (8 * j)) & 0xFF);
            bias[qb][j] = lds_f32(s.tab + min(p, s.npos - 1) * 4);
          }
        }
      if ((special >> kb) & 1) {
        unsigned cls = 0;
        if constexpr (PATH != PATH_PAIR) cls = lds_u32(s.kcls + key0);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int c = (cls >> (8 * j)) & 0xFF;
          const bool dead = PATH == PATH_PAIR ? key0 + j >= L : c == KEY_DEAD;
#pragma unroll
          for (int qb = 0; qb < QB; ++qb) {
            if constexpr (PATH != PATH_PAIR) {
              const float ct = w.qtok[qb] ? s.tokb[1] : bias[qb][j];
              const float tt = w.qtok[qb] ? s.tokb[2] : s.tokb[0];
              bias[qb][j] = c == KEY_TOKEN ? tt : ct;
            }
            // dead keys' K rows are zero, so this is their score: exp2 of it is 0
            // against any offset (offsets are real scores)
            if (dead) bias[qb][j] = AST_NEG_BIG;
          }
        }
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) v[qb][kb][j] = fmaf(v[qb][kb][j], scale, bias[qb][j]);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // largest score of each query in this lane; whether any offset has to move
  float mx[QB];
  auto over = [&]() -> bool {
    bool bad = false;
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      float t = v[qb][0][0];
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
        for (int j = 0; j < 4; ++j) t = fmaxf(t, v[qb][kb][j]);
      mx[qb] = t;
      bad |= t > 0.f || !(w.l[qb][0] > 0.f);
    }
    return __builtin_amdgcn_ballot_w64(bad) != 0;
  };
  // moves them; whether one fell far. Queries whose offset stays (delta 0) keep their
  // bits, whatever the others of the wave do.
  bool drop[QB];
  auto shift = [&]() -> bool {
    bool far = false;
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      const float g = max_groups_swap(mx[qb]), m0 = fabsf(w.m[qb]);
      const bool seen = w.l[qb][0] > 0.f;
      // no live key yet: the offset goes to this block's maximum, if it has one
      const float delta = seen ? fmaxf(g, 0.f) : (g > 0.1f * AST_NEG_BIG ? g : 0.f);
      const float alpha = seen ? __builtin_amdgcn_exp2f(-delta) : 0.f;
      w.m[qb] += delta;
      drop[qb] = m0 > FAR_OFFSET && m0 > 2.f * fabsf(w.m[qb]);
      far |= drop[qb];
      const float c = -w.m[qb] * s.inv_scale, lsum = w.l[qb][0] * alpha;
      w.cinit[qb] = f32x4{c, c, c, c};
      w.l[qb] = f32x4{lsum, lsum, lsum, lsum};
#pragma unroll
      for (int kd = 0; kd < KD; ++kd) w.o[qb][kd] = w.o[qb][kd] * alpha;
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
        for (int j = 0; j < 4; ++j) v[qb][kb][j] -= delta;
    }
    return __builtin_amdgcn_ballot_w64(far) != 0;
  };
  score();
  if (over()) {
    bool far = shift();
    // Scores formed as score - m carry m's rounding, so an offset far larger than the
    // one that replaces it (a first chunk of keys masked by -1e9, say) leaves them
    // without their digits: -1e9 in a pair table gave errors of 0.5. They are formed
    // again around the new one.
#pragma unroll 1
    for (int n = 0; __builtin_expect(far, 0) && n < MAX_RESCORES; ++n) {
      f32x4 keep[QB][NKB];
#pragma unroll
      for (int qb = 0; qb < QB; ++qb)
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb) keep[qb][kb] = v[qb][kb];
      score();
#pragma unroll
      for (int qb = 0; qb < QB; ++qb)
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb) v[qb][kb] = drop[qb] ? v[qb][kb] : keep[qb][kb];
      (void)over();
      far = shift();
    }
  }
  u32x2 pf[QB][NKB], pl[QB][FINE ? NKB : 1];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb)
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb) {
      float p[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) p[j] = __builtin_amdgcn_exp2f(v[qb][kb][j]);
      if constexpr (FINE) {
        // high part cut, not rounded, and below the weight: the low part is positive,
        // so an infinite value of V stays one (0 or less times it would be a NaN)
        unsigned t[4];
        float r[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          t[j] = __float_as_uint(p[j] * (1.f - 0x1p-16f));
          r[j] = p[j] - __uint_as_float(t[j] & 0xFFFF0000u);
        }
        pf[qb][kb] = u32x2{__builtin_amdgcn_perm(t[1], t[0], 0x07060302u),
                           __builtin_amdgcn_perm(t[3], t[2], 0x07060302u)};
        pl[qb][kb] = u32x2{pack_bf16x2(r[0], r[1]), pack_bf16x2(r[2], r[3])};
      } else {
        pf[qb][kb] = u32x2{pack_bf16x2(p[0], p[1]), pack_bf16x2(p[2], p[3])};
      }
    }
  __builtin_amdgcn_sched_barrier(0);
  const unsigned one2 = 0x3F803F80u;
  const int vrow = 4 * lg + (lr >> 2);
  const int vsw = swz<D>(vrow);
  const int vlane = vbuf + vrow * RB + (lr & 1) * 8;
#pragma unroll
  for (int kp = 0; kp < NKB; kp += 2) {
    u32x4 pp[QB], pm[QB];
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      pp[qb] = u32x4{pf[qb][kp].x, pf[qb][kp].y, pf[qb][kp + 1].x, pf[qb][kp + 1].y};
      w.l[qb] = mfma16x16x32(u32x4{one2, one2, one2, one2}, pp[qb], w.l[qb]);
      if constexpr (FINE) {
        pm[qb] = u32x4{pl[qb][kp].x, pl[qb][kp].y, pl[qb][kp + 1].x, pl[qb][kp + 1].y};
        w.l[qb] = mfma16x16x32(u32x4{one2, one2, one2, one2}, pm[qb], w.l[qb]);
      }
    }
    int at[KD];
    u32x2 v0[KD], v1[KD];
#pragma unroll
    for (int kd = 0; kd < KD; ++kd)
      at[kd] = vlane + kp * 16 * RB + (((kd * 2 + ((lr & 3) >> 1)) ^ vsw) << 4);
    lds_tr<16 * RB>(at, v0, v1);
#pragma unroll
    for (int kd = 0; kd < KD; ++kd)
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        const u32x4 vf{v0[kd].x, v0[kd].y, v1[kd].x, v1[kd].y};
        w.o[qb][kd] = mfma16x16x32(vf, pp[qb], w.o[qb][kd]);
        if constexpr (FINE) w.o[qb][kd] = mfma16x16x32(vf, pm[qb], w.o[qb][kd]);
      }
  }
}

// LDS layout (bytes): [K, V chunk 0][K, V chunk 1][tables][kkey 4 SC or kqr 8 SC]
// [kcls SC][flags][span per wave], SC = S rounded up to whole chunks; coords mode
// only past the tables. All of it dynamic, so stream_smem is what a launch needs.
// 51.7 KB at D = 64 and S = 584: three workgroups per compute unit.
__host__ __device__ inline int stream_keys(int S) { return (S + KC - 1) / KC * KC; }
__host__ __device__ inline int stream_flag_bytes(int SC) { return (SC / KC + 15) / 16 * 16; }
constexpr int SPAN_BYTES = 4 * 4 * 4;
__host__ __device__ inline int stream_tab_bytes(bool pair, int npos) {
  return pair ? (npos * 4 + 15) / 16 * 16 : (MAX_OFFSETS * 4 + 15) / 16 * 16;
}

template <int D, int QB, bool PAIR, bool FINE>
__global__ __launch_bounds__(256, QB == 2 ? 3 : 4) void attn_stream_kernel(const shrimp_attn_args a, float scale,
                                                             uint32_t qkv_bytes, int npos,
                                                             uint32_t o_bytes, int tiles) {
  constexpr int KS = D / 32, KD = D / 16, RB = 2 * D;
  constexpr int CB = KC * RB;         // bytes of one chunk's K (or V) rows
  constexpr int PPR = D / 8;          // 16-byte pieces per row
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

  // consecutive ids on one XCD (workgroups are dealt to the 8 XCDs round-robin),
  // so the query tiles of a (position, head) read K and V through one L2
  const int n = (int)gridDim.x;
  const int xcd = (int)blockIdx.x & 7, nq = n >> 3, nr = n & 7;
  const int id = xcd * nq + min(xcd, nr) + ((int)blockIdx.x >> 3);
  const int bh = id / tiles, tile = id - bh * tiles;
  const int b = bh / a.H, h = bh - b * a.H;

  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  const int lr = lane & 15, lg = lane >> 4;
  const int S = a.S, SC = stream_keys(S), nt = a.n_tokens, NC = S - nt, H = a.H;
  int L = a.seq_lens[b];
  SHRIMP_DCHECK(L >= 0 && L <= S, SHRIMP_DBG_SEQ_LEN);
  L = L < 0 ? 0 : (L > S ? S : L);

  const __amdgpu_buffer_rsrc_t ors = make_rsrc(a.o, o_bytes);
  const int qw = tile * (64 * QB) + wave * (16 * QB);  // the wave's first query
  StreamQuery<D, QB> w;
  auto store = [&]() {
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      const int query = qw + qb * 16 + lr;
      const bool on = query < L;
      const float inv = on && w.l[qb][0] > 0.f ? 1.0f / w.l[qb][0] : 0.f;
      const int64_t orow = (int64_t)b * a.o_sb + (int64_t)h * a.o_sh + (int64_t)query * a.o_sr;
#pragma unroll
      for (int kd = 0; kd < KD; ++kd) {
        const int e = kd * 16 + lg * 4;
        u32x2 pk;
        pk.x = pack_bf16x2(w.o[qb][kd][0] * inv, w.o[qb][kd][1] * inv);
        pk.y = pack_bf16x2(w.o[qb][kd][2] * inv, w.o[qb][kd][3] * inv);
        if (!on) pk = u32x2{0u, 0u};
        __builtin_amdgcn_raw_buffer_store_b64(
            pk, ors, query < S && e < a.d ? (uint32_t)((orow + e) * 2) : SHRIMP_OOB_OFFSET, 0, 0);
      }
    }
  };
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    w.m[qb] = 0.f;
    w.l[qb] = w.cinit[qb] = f32x4{0.f, 0.f, 0.f, 0.f};
    w.qkey[qb] = w.qq[qb] = w.qr[qb] = 0;
    w.qtok[qb] = qw + qb * 16 + lr < nt;
#pragma unroll
    for (int kd = 0; kd < KD; ++kd) w.o[qb][kd] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  if (tile * (64 * QB) >= L) {  // uniform: only rows past the bound
    store();
    return;
  }

  unsigned char* tabs = smem + 4 * CB;
  int2* kqr = reinterpret_cast<int2*>(tabs + stream_tab_bytes(PAIR, npos));
  int* kkey = reinterpret_cast<int*>(kqr);
  unsigned char* kcls = reinterpret_cast<unsigned char*>(kqr + SC);
  unsigned char* flags = kcls + SC;  // per chunk: bit kb, key block kb holds a token or dead key
  int(*span_red)[4] = reinterpret_cast<int(*)[4]>(flags + stream_flag_bytes(SC));

  const int64_t base = (int64_t)b * a.qkv_sb + (int64_t)h * a.qkv_sh;
  const __amdgpu_buffer_rsrc_t qrs = make_rsrc(a.q, qkv_bytes);
  const __amdgpu_buffer_rsrc_t krs = make_rsrc(a.k, qkv_bytes);
  const __amdgpu_buffer_rsrc_t vrs = make_rsrc(a.v, qkv_bytes);
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const int query = qw + qb * 16 + lr;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      w.qf[qb][ks] = buf_load16(
          qrs, query < L ? (uint32_t)((base + query * D + ks * 32 + lg * 8) * 2) : SHRIMP_OOB_OFFSET);
  }

  // 1 KiB DMAs of a chunk's K, then V rows: lane -> (row, slot), the slot's
  // piece by the row's swizzle; dead keys land as zeros
  auto dma = [&](int c, int buf) {
#pragma unroll
    for (int i = 0; i < 2 * PPR / 4; ++i) {
      const int j = wave + 4 * i;
      const int tensor = j >= PPR ? 1 : 0;
      const int row = (j - tensor * PPR) * (64 / PPR) + lane / PPR;
      const int piece = (lane % PPR) ^ swz<D>(row);
      const int key = c * KC + row;
      const bool ok = PAIR ? key < L : lds_u8(lds_addr(kcls) + key) != KEY_DEAD;
      const uint32_t off =
          ok ? (uint32_t)((base + (int64_t)key * D + piece * 8) * 2) : SHRIMP_OOB_OFFSET;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(tensor ? vrs : krs,
                                               (lds_dst_t*)(smem + buf * 2 * CB + j * 1024), 16, off,
                                               0, 0, 0);
    }
  };
  StreamLds s;
  s.keys = lds_addr(kqr);
  s.kcls = lds_addr(kcls);
  s.tab = lds_addr(tabs);
  s.npos = npos;
  s.inv_scale = 1.0f / scale;
  bool linear = false;
  if constexpr (PAIR) {
    for (int i = tid; i < npos; i += 256)
      reinterpret_cast<float*>(tabs)[i] = a.table2[(int64_t)i * H + h] * AST_LOG2E;
  } else {
    // key classes and coordinates, span of the live cells
    int qmin = 1 << 30, qmax = -(1 << 30), rmin = 1 << 30, rmax = -(1 << 30);
    for (int key = tid; key < SC; key += 256) {
      int q = 0, r = 0, cls = KEY_DEAD;  // keys past the bound (tokens too) are dead
      if (key < nt && key < L) {
        cls = KEY_TOKEN;
      } else if (key >= nt && key < L) {
        const int64_t cell = (int64_t)b * NC + (key - nt);
        q = a.coords[cell * 2];
        r = a.coords[cell * 2 + 1];
        cls = a.mask[cell] != 0 ? KEY_CELL : KEY_DEAD;
        if (cls == KEY_CELL) {
          qmin = min(qmin, q);
          qmax = max(qmax, q);
          rmin = min(rmin, r);
          rmax = max(rmax, r);
        }
      }
      kcls[key] = (unsigned char)cls;
      // a wave covers one whole chunk per iteration
      const uint64_t sp = __builtin_amdgcn_ballot_w64(cls != KEY_CELL);
      if (lane == 0)
        flags[key / KC] = (unsigned char)(((sp & 0xFFFFu) != 0) | ((sp >> 16 & 0xFFFFu) != 0) << 1 |
                                          ((sp >> 32 & 0xFFFFu) != 0) << 2 | ((sp >> 48) != 0) << 3);
    }
    for (int m = 32; m >= 1; m >>= 1) {
      qmin = min(qmin, __shfl_xor(qmin, m, 64));
      qmax = max(qmax, __shfl_xor(qmax, m, 64));
      rmin = min(rmin, __shfl_xor(rmin, m, 64));
      rmax = max(rmax, __shfl_xor(rmax, m, 64));
    }
    if (lane == 0) {
      span_red[wave][0] = qmin;
      span_red[wave][1] = qmax;
      span_red[wave][2] = rmin;
      span_red[wave][3] = rmax;
    }
    const int W2 = (2 * a.lut_m + 1) * (2 * a.lut_m + 1);
#pragma unroll
    for (int i = 0; i < 3; ++i) s.tokb[i] = a.btab[(int64_t)(W2 + i) * H + h];
    __syncthreads();
    dma(0, 0);  // under the table's round trip
    int q0 = span_red[0][0], q1 = span_red[0][1], r0 = span_red[0][2], r1 = span_red[0][3];
#pragma unroll
    for (int i = 1; i < 4; ++i) {
      q0 = min(q0, span_red[i][0]);
      q1 = max(q1, span_red[i][1]);
      r0 = min(r0, span_red[i][2]);
      r1 = max(r1, span_red[i][3]);
    }
    // LINEAR needs a live cell (token and dead keys borrow its code) and the
    // spanned offsets to fit the table region
    const int64_t sq = (int64_t)q1 - q0, sr = (int64_t)r1 - r0;
    linear = sq >= 0 && sq < MAX_OFFSETS && sr < MAX_OFFSETS &&
             (2 * sq + 1) * (2 * sr + 1) <= MAX_OFFSETS;
    const int M = a.lut_m, W = 2 * M + 1, XW = linear ? 2 * (int)sr + 1 : 0;
    float* tab = reinterpret_cast<float*>(tabs);
    if (linear) {
      // a wave per row of offsets dq, lanes along dr; a thread's loads all issued
      // before its stores (one by one they cost 14 round trips, 5 us per workgroup)
      for (int c0 = 0; c0 < XW; c0 += 64) {
        const int dr = c0 + lane;
        const int col = (clampi(dr - (int)sr, M) + M) * H + h;
        for (int d0 = wave; d0 <= 2 * (int)sq; d0 += 4 * TU) {
          float t[TU];
#pragma unroll
          for (int u = 0; u < TU; ++u) {
            const int dq = min(d0 + 4 * u, 2 * (int)sq);
            t[u] = a.btab[(int64_t)(clampi(dq - (int)sq, M) + M) * W * H + col];
          }
#pragma unroll
          for (int u = 0; u < TU; ++u)
            if (dr < XW && d0 + 4 * u <= 2 * (int)sq) tab[(d0 + 4 * u) * XW + dr] = t[u];
        }
      }
    } else {
      for (int i = tid; i < W2; i += 256) tab[i] = a.btab[(int64_t)i * H + h];
    }
    // LINEAR: token and dead keys take the code of the live cell (q0, r0), so
    // every read stays inside the table; their biases are selected afterwards
    const int xoff = lds_addr(tabs) + (linear ? ((int)sq * XW + (int)sr) * 4 : 0);
    auto code = [&](int2 c) { return ((c.x - q0) * XW + (c.y - r0)) * 4; };
    auto cell_of = [&](int key) {
      const int64_t cell = (int64_t)b * NC + (key - nt);
      return make_int2(a.coords[cell * 2], a.coords[cell * 2 + 1]);
    };
    for (int key = tid; key < SC; key += 256) {
      const bool cell = kcls[key] == KEY_CELL;
      if (linear) kkey[key] = xoff + (cell ? code(cell_of(key)) : 0);
      else kqr[key] = cell ? cell_of(key) : make_int2(0, 0);
    }
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      const int query = qw + qb * 16 + lr;
      w.qq[qb] = w.qr[qb] = w.qkey[qb] = 0;
      if (query < L && kcls[query] == KEY_CELL) {
        const int2 c = cell_of(query);
        w.qq[qb] = c.x;
        w.qr[qb] = c.y;
        if (linear) w.qkey[qb] = code(c);
      }
    }
  }

  // pair rows of a chunk: four table rows per 16-key block and lane
  unsigned pn[QB][4];
  auto load_pair = [&](int c, unsigned (&p)[QB][4]) {
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      const int query = qw + qb * 16 + lr;
      const uint8_t* row = a.pair + (int64_t)b * a.p_sb + (int64_t)(query < L ? query : 0) * a.p_sq;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        const int key = c * KC + kb * 16 + lg * 4;
        unsigned x = 0;
        if (c * KC + KC <= S) {
          __builtin_memcpy(&x, row + key, 4);
        } else if (S >= 4) {  // past the row's end: its last four keys, shifted
          const int at = min(key, S - 4);
          __builtin_memcpy(&x, row + at, 4);
          x = key - at < 4 ? x >> (8 * (key - at)) : 0u;
        } else {
          for (int j = 0; j < 4; ++j)
            if (key + j < S) x |= (unsigned)row[key + j] << (8 * j);
        }
        p[qb][kb] = x;
      }
    }
  };
#pragma unroll
  for (int qb = 0; qb < QB; ++qb)
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) pn[qb][kb] = 0;

  const int nc = (L + KC - 1) / KC;
  const bool active = qw < L;
  const bool tok = !PAIR && qw < nt;  // the wave's queries hold tokens
  const int lds0 = lds_addr(smem);
  if (PAIR) dma(0, 0);
  if (PAIR && active) load_pair(0, pn);
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  // one loop per bias path: the paths share no registers
  auto run = [&](auto path) {
    for (int c = 0; c < nc; ++c) {
      const int buf = c & 1;
      unsigned pd[QB][4];
      if constexpr (PAIR) {
#pragma unroll
        for (int qb = 0; qb < QB; ++qb)
#pragma unroll
          for (int kb = 0; kb < 4; ++kb) pd[qb][kb] = pn[qb][kb];
      }
      if (c + 1 < nc) {
        dma(c + 1, buf ^ 1);
        if (PAIR && active) load_pair(c + 1, pn);
      }
      if (active) {
        const int kbuf = lds0 + buf * 2 * CB, vbuf = kbuf + CB;
        int special;
        if constexpr (PAIR) {
          const int over = L - c * KC;  // keys of the chunk inside the bound
          special = over >= KC ? 0 : (15 << (over >> 4)) & 15;
        } else {
          special = tok ? 15 : __builtin_amdgcn_readfirstlane((int)lds_u8(lds_addr(flags) + c));
        }
        constexpr int NKB = stream_nkb<decltype(path)::value>();
#pragma unroll 1
        for (int kb = 0; kb < 4 && c * KC + kb * 16 < L; kb += NKB) {
          unsigned p[QB][NKB];
          if constexpr (PAIR) {
#pragma unroll
            for (int qb = 0; qb < QB; ++qb)
#pragma unroll
              for (int i = 0; i < NKB; ++i) p[qb][i] = pd[qb][i];
          }
          stream_chunk<D, QB, decltype(path)::value, FINE>(
              a, w, s, c * KC + kb * 16, L, special >> kb, kbuf + kb * 16 * RB, vbuf + kb * 16 * RB,
              lr, lg, scale, p);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
    }
  };
  if constexpr (PAIR) {
    run(std::integral_constant<int, PATH_PAIR>{});
  } else {
    if (linear) run(std::integral_constant<int, PATH_LINEAR>{});
    else run(std::integral_constant<int, PATH_CLAMP>{});
  }
  store();
}

size_t stream_smem(int D, bool pair, int S, int npos) {
  const size_t SC = (size_t)stream_keys(S);
  return (size_t)4 * KC * 2 * D + stream_tab_bytes(pair, npos) +
         (pair ? 0 : SC * 9 + stream_flag_bytes((int)SC) + SPAN_BYTES);
}

}  // namespace

// Whether the streamed kernel covers the call: padded head dim 32 or 64, q / k
// / v rows on 16-byte boundaries (DMA pieces), tables within a workgroup's LDS.
bool attn_stream_ok(const shrimp_attn_args* a, int npos) {
  if (a->dpad != 32 && a->dpad != 64) return false;
  const uintptr_t p = reinterpret_cast<uintptr_t>(a->q) | reinterpret_cast<uintptr_t>(a->k) |
                      reinterpret_cast<uintptr_t>(a->v);
  if ((p & 15) != 0 || a->qkv_sb % 8 != 0 || a->qkv_sh % 8 != 0) return false;
  if (a->pair == nullptr && a->lut_m > MAX_LUT_M) return false;
  if ((int64_t)a->B * a->H * ((a->S + 63) / 64) >= (1 << 30)) return false;
  return stream_smem(a->dpad, a->pair != nullptr, a->S, npos) <= (size_t)max_lds_per_block();
}

template <int D, int QB, bool PAIR, bool FINE>
static int launch_stream(const shrimp_attn_args* a, float scale, uint32_t qkv_bytes, int npos,
                         uint32_t o_bytes, hipStream_t st) {
  const int tiles = (a->S + 64 * QB - 1) / (64 * QB);
  hipLaunchKernelGGL((attn_stream_kernel<D, QB, PAIR, FINE>), dim3(a->B * a->H * tiles), dim3(256),
                     stream_smem(D, PAIR, a->S, npos), st, *a, scale, qkv_bytes, npos, o_bytes, tiles);
  return check_launch("attn");
}

// Coords: 32 queries per wave (each K and V fragment read feeds two products) past 64
// rows once such tiles give every compute unit two workgroups, else 16, with the same
// bits. Measured at 768 positions, H = 4, D = 32, 16 against 32: 200 rows 1.27 times the
// time, 328 rows 1.32, 64 rows (half of a 128-query tile empty) 0.88. Pair: 16, whose
// scores wait for their pair rows (32 against them from 104 rows 0.97 to 1.41 times the
// time; at 72 rows, 512 positions, H = 4, D = 32 22.6 us for 26.7, left for one set of
// bits at every batch). fine: weights as two bf16 numbers, their product with V as
// two (dispatch_attn says where).
int launch_attn_stream(const shrimp_attn_args* a, float scale, uint32_t qkv_bytes, int npos,
                       uint32_t o_bytes, bool fine, hipStream_t st) {
  const bool wide = a->S > 64 && (int64_t)a->B * a->H * ((a->S + 127) / 128) >= 2 * cu_count();
#define AST_LAUNCH(...)                                                                       \
  do {                                                                                        \
    if (fine) return launch_stream<__VA_ARGS__, true>(a, scale, qkv_bytes, npos, o_bytes, st); \
    return launch_stream<__VA_ARGS__, false>(a, scale, qkv_bytes, npos, o_bytes, st);         \
  } while (0)
  if (a->dpad == 64) {
    if (a->pair != nullptr) AST_LAUNCH(64, 1, true);
    if (wide) AST_LAUNCH(64, 2, false);
    AST_LAUNCH(64, 1, false);
  }
  if (a->pair != nullptr) AST_LAUNCH(32, 1, true);
  if (wide) AST_LAUNCH(32, 2, false);
  AST_LAUNCH(32, 1, false);
#undef AST_LAUNCH
}

}  // namespace shrimp
