// The bf16 trunk of one forward (stem, blocks, tail, heads) as one call: the
// launch sequence of HipForward._trunk (shrimp/runtime.py; reference
// model.py:395-514, 865, 905-1020) issued from native code. A network of 12
// blocks is about 40 launches; building each one's arguments in Python took
// 8-10 us, more than most kernels of a small batch run for.
//
// Host code only: every launch goes through the entry points of the C ABI, with
// their argument checks, on the caller's stream and in the caller's workspace.
#include <cstring>

#include "capi.hpp"

namespace {

// Network words (int64, host memory; pointers to device memory, eps as float bits).
enum : int {
  W_LAYERS, W_C, W_H, W_D, W_DPAD, W_TOKENS, W_STEM_W, W_STEM_B, W_STEM_LNW, W_STEM_LNB, W_STEM_EPS,
  W_LNF_W, W_LNF_B, W_LNF_EPS, W_VALUE,  // four head pointers each: rw, rb, hw, hb
  W_ML = W_VALUE + 4, W_POLICY_W = W_ML + 4, W_POLICY_B, W_POLICY_HW, W_POLICY_HB,
  W_LUT_M, W_TOKEN_ROWS, W_BINS, W_HEAD_END
};
// Per layer: kind (0 ConvBlock, 1 AttnBlock), then
enum : int { L_KIND, L_WORDS = 21 };
enum : int { C_W1 = 1, C_B1, C_LN1W, C_LN1B, C_EPS1, C_W2, C_B2, C_LN2W, C_LN2B, C_EPS2, C_GAMMA };
enum : int { A_QKV = 1, A_QKV_W, A_QKV_B, A_LN1W, A_LN1B, A_EPS1, A_MLP, A_OUT_W, A_OUT_B, A_GATTN,
             A_LN2W, A_LN2B, A_EPS2, A_FC1_W, A_FC1_B, A_FC2_W, A_FC2_B, A_GMLP, A_BTAB, A_XTAB };
// Call words.
enum : int { I_IDX, I_MASK8, I_COORDS, I_SEQ_LENS, I_SEQ_MASK, I_XIN, I_WORKSPACE, I_QKV, I_POLICY,
             I_VALUE, I_ML, I_B, I_N, I_FLAGS, I_WORDS };
enum : int { F_STAGED = 1, F_QKV = 2, F_MLP = 4, F_BLOCK = 8, F_PAIR = 16, F_TAIL = 32, F_LINEAR_BIAS = 64,
             F_END = 128 };

float bits(int64_t w) {
  const uint32_t u = (uint32_t)w;
  float f;
  std::memcpy(&f, &u, 4);
  return f;
}
template <class T = void>
const T* cp(int64_t w) {
  return reinterpret_cast<const T*>((uintptr_t)w);
}
template <class T = void>
T* mp(int64_t w) {
  return reinterpret_cast<T*>((uintptr_t)w);
}

// Workspace regions, 256-byte aligned.
struct Regions {
  int64_t seq, tok_lo, y1, qkv, att, hid, kvf, meta, seqf, tail, total;
};

Regions regions(const int64_t* net, int64_t B, int64_t N, int flags, bool own_qkv) {
  const int64_t C = net[W_C], H = net[W_H], dpad = net[W_DPAD], nt = net[W_TOKEN_ROWS], S = N + nt;
  const int64_t SP = (S + 15) / 16 * 16;
  const bool staged = (flags & F_STAGED) != 0;
  Regions r{};
  int64_t at = 0;
  auto take = [&](int64_t bytes) {
    const int64_t here = at;
    at += (bytes + 255) / 256 * 256;
    return here;
  };
  r.seq = take(B * S * C * 2);
  r.tok_lo = take(B * nt * C * 2);
  r.y1 = take(flags & F_BLOCK ? 0 : B * N * C * 2);
  r.qkv = take(own_qkv ? (staged ? 1 : 3) * B * H * S * dpad * 2 : 0);
  r.att = take(B * S * C * 2);
  r.hid = take(flags & F_MLP ? 0 : B * S * 4 * C);
  r.kvf = take(staged ? B * H * SP * 64 : 0);
  r.meta = take(staged ? B * (int64_t)shrimp_attn_keys_bytes((int)S) : 0);
  r.seqf = take(flags & F_TAIL ? 0 : B * S * C * 2);
  r.tail = take(B * 6 * C * 4);
  r.total = at;
  return r;
}

// Everything that is narrowed to int below, and row counts, inside int.
bool shape_ok(const int64_t* net, int64_t B, int64_t N, int64_t flags) {
  const int64_t c = net[W_C], h = net[W_H], d = net[W_D], dp = net[W_DPAD], nt = net[W_TOKEN_ROWS];
  return B > 0 && N > 0 && N < shrimp::kMaxDim && flags >= 0 && flags < F_END && c > 0 && c <= 4096 &&
         h > 0 && c % h == 0 && c / h == d && dp >= d && dp <= 4096 && nt > 0 && nt <= 4096 &&
         net[W_LUT_M] >= 0 && net[W_LUT_M] <= 64 && net[W_BINS] > 0 && net[W_BINS] <= 4096 &&
         shrimp::mul_sat({B, N + nt}) <= INT32_MAX &&
         shrimp::mul_sat({B, N + nt, 4, c > h * dp ? c : h * dp, 2}) < ((int64_t)1 << 40);
}

}  // namespace

extern "C" int64_t shrimp_forward_bytes(const int64_t* net, int B, int N, int flags, int own_qkv) {
  if (net == nullptr || !shape_ok(net, B, N, flags)) return 0;
  return regions(net, B, N, flags, own_qkv != 0).total;
}

extern "C" int shrimp_forward(const int64_t* net, const int64_t* io, void* stream) {
  SHRIMP_REQUIRE(net && io, "forward: null words");
  if (io[I_B] == 0) return SHRIMP_OK;
  SHRIMP_REQUIRE(shape_ok(net, io[I_B], io[I_N], io[I_FLAGS]) && net[W_LAYERS] > 0 &&
                     net[W_LAYERS] <= 1 << 20,
                 "forward: bad shape (B %lld, N %lld, C %lld, H %lld, d %lld, flags %lld)",
                 (long long)io[I_B], (long long)io[I_N], (long long)net[W_C], (long long)net[W_H],
                 (long long)net[W_D], (long long)io[I_FLAGS]);
  for (int64_t i = 0; i < net[W_LAYERS]; ++i)
    SHRIMP_REQUIRE((net[W_HEAD_END + i * L_WORDS + L_KIND] | 1) == 1, "forward: layer %d of kind %lld",
                   (int)i, (long long)net[W_HEAD_END + i * L_WORDS + L_KIND]);
  SHRIMP_REQUIRE(net[W_TOKENS] != 0 && io[I_SEQ_MASK] != 0, "forward: null tokens or sequence mask");
  SHRIMP_REQUIRE(io[I_WORKSPACE] != 0 && (io[I_WORKSPACE] & 255) == 0,
                 "forward: workspace must be 256-byte aligned");
  const int B = (int)io[I_B], N = (int)io[I_N], flags = (int)io[I_FLAGS];
  const int C = (int)net[W_C], H = (int)net[W_H], d = (int)net[W_D], dpad = (int)net[W_DPAD];
  const int nt = (int)net[W_TOKEN_ROWS], S = N + nt, rows = B * S, lut_m = (int)net[W_LUT_M];
  const Regions r = regions(net, B, N, flags, io[I_QKV] == 0);
  unsigned char* ws = mp<unsigned char>(io[I_WORKSPACE]);
  void* seq = ws + r.seq;
  void* cells = ws + r.seq + (int64_t)nt * C * 2;
  void* tok_lo = ws + r.tok_lo;
  void* y1 = ws + r.y1;
  uint16_t* qkv = io[I_QKV] ? mp<uint16_t>(io[I_QKV]) : reinterpret_cast<uint16_t*>(ws + r.qkv);
  void* att = ws + r.att;
  void* hid = ws + r.hid;
  int32_t* meta = reinterpret_cast<int32_t*>(ws + r.meta);
  const int32_t* idx = cp<int32_t>(io[I_IDX]);
  const uint8_t* mask8 = cp<uint8_t>(io[I_MASK8]);
  const int32_t* coords = cp<int32_t>(io[I_COORDS]);
  const int32_t* seq_lens = cp<int32_t>(io[I_SEQ_LENS]);
  const uint8_t* seq_mask = cp<uint8_t>(io[I_SEQ_MASK]);
  const int64_t sb = (int64_t)S * C, plane = (int64_t)B * H * S * dpad;
  const bool staged = (flags & F_STAGED) != 0;
#define FWD(call)                      \
  do {                                 \
    if (int rc = (call)) return rc;    \
  } while (0)

  if (staged)
    FWD(shrimp_attn_keys_tokens(coords, mask8, seq_lens, B, S, nt, meta, cp<float>(net[W_TOKENS]), C,
                                seq, sb, tok_lo, stream));
  else
    FWD(shrimp_fill_tokens(cp<float>(net[W_TOKENS]), nt, C, seq, sb, tok_lo, B, stream));

  auto conv = [&](const void* x, int64_t x_sb, int64_t x_sn, int64_t w, int64_t b, int cin_pad) {
    shrimp_conv_args a{};
    a.x = x;
    a.x_sb = x_sb;
    a.x_sn = x_sn;
    a.idx = idx;
    a.taps = 7;
    a.idx_stride = 7;
    a.mask = mask8;
    a.w = cp(w);
    a.bias = cp<float>(b);
    a.eps = 1e-5f;
    a.B = B;
    a.N = N;
    a.cin_pad = cin_pad;
    a.cout = C;
    return a;
  };
  auto norm = [&](shrimp_conv_args& a, int64_t w, int64_t b, int64_t eps) {
    a.ln_w = cp<float>(w);
    a.ln_b = cp<float>(b);
    a.eps = bits(eps);
  };
  auto to_cells = [&](shrimp_conv_args& a) {
    a.out = cells;
    a.o_sb = sb;
    a.o_sn = C;
  };
  {
    shrimp_conv_args a = conv(cp(io[I_XIN]), (int64_t)N * 32, 32, net[W_STEM_W], net[W_STEM_B], 32);
    norm(a, net[W_STEM_LNW], net[W_STEM_LNB], net[W_STEM_EPS]);
    a.relu = 1;
    to_cells(a);
    FWD(shrimp_hex_conv(&a, stream));
  }
  // the two convs of ConvBlock l, reading and writing the cell rows in place
  auto first = [&](const int64_t* l) {
    shrimp_conv_args a = conv(cells, sb, C, l[C_W1], l[C_B1], C);
    norm(a, l[C_LN1W], l[C_LN1B], l[C_EPS1]);
    a.relu = 1;
    return a;
  };
  auto second = [&](const int64_t* l, const void* x, int64_t x_sb) {
    shrimp_conv_args a = conv(x, x_sb, C, l[C_W2], l[C_B2], C);
    norm(a, l[C_LN2W], l[C_LN2B], l[C_EPS2]);
    a.resid = cells;
    a.r_sb = sb;
    a.r_sn = C;
    a.gamma = cp<float>(l[C_GAMMA]);
    to_cells(a);
    return a;
  };
  const int64_t* layers = net + W_HEAD_END;
  const int n_layers = (int)net[W_LAYERS];
  for (int i = 0; i < n_layers; ++i) {
    const int64_t* l = layers + (int64_t)i * L_WORDS;
    if (l[L_KIND] == 0) {
      if ((flags & F_PAIR) && i + 1 < n_layers && l[L_WORDS + L_KIND] == 0) {
        const int64_t* m = l + L_WORDS;
        shrimp_conv_args c1 = first(l), c2 = second(l, cells, sb), c3 = first(m),
                         c4 = second(m, cells, sb);
        FWD(shrimp_conv_block_pair(&c1, &c2, &c3, &c4, stream));
        ++i;
      } else if (flags & F_BLOCK) {
        shrimp_conv_args c1 = first(l), c2 = second(l, cells, sb);
        FWD(shrimp_conv_block(&c1, &c2, stream));
      } else {
        shrimp_conv_args c1 = first(l);
        c1.out = y1;
        c1.o_sb = (int64_t)N * C;
        c1.o_sn = C;
        FWD(shrimp_hex_conv(&c1, stream));
        shrimp_conv_args c2 = second(l, y1, (int64_t)N * C);
        FWD(shrimp_hex_conv(&c2, stream));
      }
      continue;
    }
    auto linear = [&](const void* x, int64_t x_sr, int64_t w, int64_t b, int n_in, int n_out, int mode,
                      void* out, int64_t o_sr) {
      shrimp_linear_args a{};
      a.x = x;
      a.x_sr = x_sr;
      a.w = cp(w);
      a.bias = cp<float>(b);
      a.eps = 1e-5f;
      a.mode = mode;
      a.out = out;
      a.o_sr = o_sr;
      a.rows = rows;
      a.in_features = n_in;
      a.out_features = n_out;
      return a;
    };
    // LN1 + q / k / v
    if (staged || (flags & F_QKV)) {
      shrimp_qkv_args q{};
      q.x = seq;
      q.x_sr = C;
      q.qkv = qkv;
      q.packed = cp(l[A_QKV]);
      q.eps = bits(l[A_EPS1]);
      q.rows = rows;
      q.B = B;
      q.S = S;
      q.H = H;
      q.C = C;
      q.dpad = dpad;
      if (staged) FWD(shrimp_attn_qkv_kvf(&q, ws + r.kvf, stream));
      else FWD(shrimp_attn_qkv(&q, stream));
    } else {
      shrimp_linear_args q =
          linear(seq, C, l[A_QKV_W], l[A_QKV_B], C, 3 * C, SHRIMP_LIN_QKV, qkv, 0);
      q.ln_w = cp<float>(l[A_LN1W]);
      q.ln_b = cp<float>(l[A_LN1B]);
      q.eps = bits(l[A_EPS1]);
      q.B = B;
      q.S = S;
      q.H = H;
      q.dpad = dpad;
      FWD(shrimp_linear(&q, stream));
    }
    // attention
    {
      shrimp_attn_args a{};
      a.q = qkv;
      a.qkv_sb = (int64_t)H * S * dpad;
      a.qkv_sh = (int64_t)S * dpad;
      a.seq_lens = seq_lens;
      a.btab = cp<float>(l[A_BTAB]);
      a.lut_m = lut_m;
      a.n_tokens = nt;
      a.o = att;
      a.o_sb = sb;
      a.o_sh = d;
      a.o_sr = C;
      a.B = B;
      a.S = S;
      a.H = H;
      a.d = d;
      a.dpad = dpad;
      if (staged) {
        a.xtab = cp(l[A_XTAB]);
        FWD(shrimp_attn_staged(&a, ws + r.kvf, meta, stream));
      } else {
        a.xtab = flags & F_LINEAR_BIAS ? cp(l[A_XTAB]) : nullptr;
        a.k = qkv + plane;
        a.v = qkv + 2 * plane;
        a.coords = coords;
        a.mask = mask8;
        FWD(shrimp_attn(&a, stream));
      }
    }
    // out_proj, MLP
    if (flags & F_MLP) {
      shrimp_mlp_args m{};
      m.x = att;
      m.x_sr = C;
      m.seq = seq;
      m.s_sr = C;
      m.mask = seq_mask;
      m.packed = cp(l[A_MLP]);
      m.eps = bits(l[A_EPS2]);
      m.rows = rows;
      m.C = C;
      m.hidden = 2 * C;
      m.tok_lo = tok_lo;
      m.S = S;
      m.n_tokens = nt;
      FWD(shrimp_attn_mlp(&m, stream));
      continue;
    }
    auto resid = [&](shrimp_linear_args a, int64_t gamma) {
      a.resid = seq;
      a.r_sr = C;
      a.gamma = cp<float>(gamma);
      a.mask = seq_mask;
      a.S = S;
      a.tok_lo = tok_lo;
      a.n_tokens = nt;
      return a;
    };
    const shrimp_linear_args o =
        resid(linear(att, C, l[A_OUT_W], l[A_OUT_B], C, C, SHRIMP_LIN_RESID, seq, C), l[A_GATTN]);
    FWD(shrimp_linear(&o, stream));
    shrimp_linear_args f1 =
        linear(seq, C, l[A_FC1_W], l[A_FC1_B], C, 2 * C, SHRIMP_LIN_GELU, hid, 2 * C);
    f1.ln_w = cp<float>(l[A_LN2W]);
    f1.ln_b = cp<float>(l[A_LN2B]);
    f1.eps = bits(l[A_EPS2]);
    FWD(shrimp_linear(&f1, stream));
    const shrimp_linear_args f2 =
        resid(linear(hid, 2 * C, l[A_FC2_W], l[A_FC2_B], 2 * C, C, SHRIMP_LIN_RESID, seq, C), l[A_GMLP]);
    FWD(shrimp_linear(&f2, stream));
  }

  shrimp_tail_args t{};
  t.seq = seq;
  t.s_sb = sb;
  t.mask = mask8;
  t.ln_w = cp<float>(net[W_LNF_W]);
  t.ln_b = cp<float>(net[W_LNF_B]);
  t.eps = bits(net[W_LNF_EPS]);
  t.out_seq = ws + r.seqf;
  t.vr_w = cp<float>(net[W_VALUE]);
  t.vr_b = cp<float>(net[W_VALUE + 1]);
  t.vh_w = cp<float>(net[W_VALUE + 2]);
  t.vh_b = cp<float>(net[W_VALUE + 3]);
  t.value = mp<float>(io[I_VALUE]);
  t.mr_w = cp<float>(net[W_ML]);
  t.mr_b = cp<float>(net[W_ML + 1]);
  t.mh_w = cp<float>(net[W_ML + 2]);
  t.mh_b = cp<float>(net[W_ML + 3]);
  t.moves_left = mp<float>(io[I_ML]);
  t.workspace = reinterpret_cast<float*>(ws + r.tail);
  t.B = B;
  t.S = S;
  t.n_tokens = nt;
  t.C = C;
  t.bins = (int)net[W_BINS];
  t.tok_lo = tok_lo;
  const bool tail = (flags & F_TAIL) != 0;
  shrimp_conv_args p = conv(tail ? cells : static_cast<void*>(ws + r.seqf + (int64_t)nt * C * 2), sb, C,
                            net[W_POLICY_W], net[W_POLICY_B], C);
  p.relu = 1;
  p.head_w = cp<float>(net[W_POLICY_HW]);
  p.head_b = cp<float>(net[W_POLICY_HB]);
  p.head_out = mp<float>(io[I_POLICY]);
  if (tail) return shrimp_policy_tail(&p, &t, stream);
  FWD(shrimp_trunk_tail(&t, stream));
  return shrimp_hex_conv(&p, stream);
#undef FWD
}
