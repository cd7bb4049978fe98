// Host-side validation of the kernel C ABI under AddressSanitizer / UBSan
// (tests/test_host_sanitizer.py builds this with `-Xarch_host -fsanitize=...`:
// the GPU sanitizer is not available here, so the host half of every
// entry point — shape checks, config tables, the guards that keep a kernel
// from being launched with operands its grid does not cover — is what runs
// instrumented).  Every call below must be REJECTED before any launch, so the
// program needs no GPU.  Prints "host_validate ok" and exits 0 on success.
#include <cstdio>

#include "../kernels/api.h"
#include "../kernels/attention_row.h"
#include "../kernels/mixer_api.h"
#include "../kernels/residual_api.h"

static int g_fail = 0;

// Rejections are negative; 0 or a positive hipError_t means a launch was
// attempted (with no GPU it fails), i.e. the guard did not catch the shape.
static void expect_reject(int rc, const char* what) {
  if (rc >= 0) {
    std::printf("NOT REJECTED: %s (rc=%d)\n", what, rc);
    ++g_fail;
  }
}

static void expect_noop(int rc, const char* what) {
  if (rc != 0) {
    std::printf("empty problem should be a no-op: %s (rc=%d)\n", what, rc);
    ++g_fail;
  }
}

static void expect_eq(int got, int want, const char* what) {
  if (got != want) {
    std::printf("%s: %d, not %d\n", what, got, want);
    ++g_fail;
  }
}

int main() {
  alignas(16) char buf[64] = {0};
  void* p = buf;
  float* f = reinterpret_cast<float*>(buf);
  int* ip = reinterpret_cast<int*>(buf);
  hipStream_t st = nullptr;
  // decoder kernels
  RowsArgs ra = {};
  ra.x_in = f, ra.x_out = f, ra.ldx = ra.ldy = 64, ra.M = 1, ra.N = 64, ra.NP = 64;
  RowsArgs rb = ra;
  rb.M = 0;
  expect_reject(dnn_rows_update(&rb, 0, 0, st), "rows M=0");
  rb = ra, rb.N = 65;
  expect_reject(dnn_rows_update(&rb, 0, 0, st), "rows N > NP");
  rb = ra, rb.NP = 20000;
  expect_reject(dnn_rows_update(&rb, 0, 0, st), "rows too wide");
  rb = ra, rb.xidx = ip, rb.xrows = 1;
  expect_reject(dnn_rows_update(&rb, 0, 0, st), "rows gathered in-place");
  expect_reject(dnn_rows_update(&ra, 0, 1, st), "rows bf16 in, fp32 operand out");
  rb = ra, rb.y2 = f;
  expect_reject(dnn_rows_update(&rb, 0, 0, st), "rows second output without a norm");
  rb = ra, rb.ys = f, rb.top = 2;
  expect_reject(dnn_rows_update(&rb, 0, 0, st), "rows of experts without places");
  double freq = 0;
  rb = ra, rb.freq = &freq;
  expect_reject(dnn_rows_update(&rb, 0, 0, st), "positions without positions");
  {
    ConvArgs c{};
    c.in = f, c.out = f, c.M = 4, c.C = 64, c.taps = 4, c.ldi = c.ldo = 64, c.nslots = 1;
    ConvArgs d = c;
    d.C = 60;
    expect_reject(dnn_conv(&d, 0, st), "conv channels % 8");
    d = c, d.ldi = 32;
    expect_reject(dnn_conv(&d, 0, st), "conv row too short");
    d = c, d.dt = f, d.la = f, d.H = 8, d.dt_col = 60;
    expect_reject(dnn_conv(&d, 0, st), "conv step sizes past the row");
    expect_reject(dnn_conv_state(&c, nullptr, 0, 0, st), "conv state of nothing");
    ScanArgs a{};
    a.M = 4, a.H = 2, a.NP = 64, a.VP = 64, a.vdim = 64, a.nent = 1, a.nslots = 1, a.qdiv = 1, a.ld = 384, a.ldy = 128;
    a.kcol = 128, a.vcol = 256, a.la_h = f, a.state = f, a.pos = reinterpret_cast<int*>(f);
    auto scan = [&](auto edit, const char* what) {
      ScanArgs b = a;
      edit(b);
      expect_reject(dnn_scan_chunks(&b, st), what);
      expect_reject(dnn_scan_steps(&b, 0, st), what);
    };
    scan([](ScanArgs& b) { b.NP = 96; }, "scan state size 96");
    scan([](ScanArgs& b) { b.vcol = 320; }, "scan values past the row");
    scan([](ScanArgs& b) { b.vdim = 65; }, "scan value size past its padding");
    scan([](ScanArgs& b) { b.la_h = nullptr; }, "scan without decays");
    scan([](ScanArgs& b) { b.nent = 0; }, "scan of nothing");
    GatedNormArgs g{};
    g.M = 1, g.n = 65, g.groups = 2, g.ldy = g.ldz = g.ldo = 128;
    expect_reject(dnn_gated_norm(&g, 0, st), "gated norm in unequal parts");
    RouteArgs r{};
    r.M = 4, r.E = r.ldl = 8, r.groups = 2, r.keep = 1, r.top = 5;
    expect_reject(dnn_route(&r, st), "route more experts than the groups hold");
    r.top = 2, r.groups = 3;
    expect_reject(dnn_route(&r, st), "route unequal groups");
    r.groups = 2, r.E = r.ldl = 512;
    expect_reject(dnn_route(&r, st), "route too many experts");
    GroupedArgs e{};
    int offs[3] = {0, 1, 2};
    e.A = e.W = e.Wsh = e.C = nullptr, e.offs = offs, e.rows = 2, e.arows = 2, e.div = 1, e.N = e.K = 64, e.E = 2;
    e.lda = e.ldc = 64;
    expect_reject(dnn_grouped_gemm(&e, st), "grouped product without weights");
    expect_reject(dnn_grouped_gemm_f32(&e, st), "fp32 grouped product without weights");
    e.Wsh = e.W = f, e.K = 48;
    expect_reject(dnn_grouped_gemm(&e, st), "grouped product K % 64");
    e.K = 64, e.ldc = 32;
    expect_reject(dnn_grouped_gemm(&e, st), "grouped product result row too short");
    QkNormArgs q{};
    q.M = 1, q.H = 2, q.G = 1, q.DK = 64, q.ldq = 128, q.nq = 128, q.nk = 64, q.ldt = 1, q.npages = 1;
    expect_reject(dnn_qk_norm(&q, 0, st), "qk norm row too short");
    q.ldq = 192, q.nk = 65;
    expect_reject(dnn_qk_norm(&q, 0, st), "qk norm of more than the projection");
    r.E = r.ldl = 8, r.group_top = 3;
    expect_reject(dnn_route(&r, st), "route groups by three experts");
    e.ldc = 64, e.offs = nullptr, e.rows = 3;
    expect_reject(dnn_grouped_gemm(&e, st), "even product of rows that do not divide");
    e.rows = 4, e.sa = 4;
    expect_reject(dnn_grouped_gemm(&e, st), "even product at unaligned operands");
  }
  rb = ra, rb.y_joined = 1, rb.y_w = f, rb.y = f;
  expect_reject(dnn_rows_update(&rb, 0, 0, st), "rows norm of a sum without rows");
  {
    PolyNormArgs a{p, f, 64, 1, 65, 1e-5f};
    expect_reject(dnn_poly_norm(&a, 0, st), "poly norm past the row");
    a.n = 64, a.w = nullptr;
    expect_reject(dnn_poly_norm(&a, 0, st), "poly norm without weights");
    PairArgs b{};
    b.M = 1, b.nslots = 1, b.buckets = 0;
    expect_reject(dnn_pair_rows(&b, st), "pair rows of no buckets");
    b.buckets = 5, b.mul_prev = -1;
    expect_reject(dnn_pair_rows(&b, st), "pair rows with a negative factor");
    ShiftArgs s{};
    s.M = 1, s.NP = s.ldx = s.ldo = 64, s.nslots = 1, s.n = 9;
    expect_reject(dnn_token_shift(&s, 0, st), "token shift of nine mixes");
    s.n = 1, s.ldx = 32;
    expect_reject(dnn_token_shift(&s, 0, st), "token shift row too short");
    DecayArgs d{};
    d.M = 1, d.N = 64, d.rank = 48, d.ldt = 64;
    expect_reject(dnn_decay(&d, 0, st), "decay rank % 32");
    d.rank = 64, d.ldt = 32;
    expect_reject(dnn_decay(&d, 1, st), "decay row too short");
    WkvArgs w{};
    w.M = 2, w.H = 2, w.NP = 64, w.dim = 64, w.nent = w.nslots = 1, w.ld = 128, w.ldy = 128;
    w.state = f, w.pos = ip, w.la = f, w.u = f;
    auto wkv = [&](auto edit, const char* what) {
      WkvArgs x = w;
      edit(x);
      expect_reject(dnn_wkv_steps(&x, 0, st), what);
      expect_reject(dnn_wkv_chunks(&x, st), what);
    };
    wkv([](WkvArgs& x) { x.NP = 96; }, "wkv head size 96");
    wkv([](WkvArgs& x) { x.dim = 65; }, "wkv head past its padding");
    wkv([](WkvArgs& x) { x.ld = 64; }, "wkv row too short");
    wkv([](WkvArgs& x) { x.u = nullptr; }, "wkv without a bonus");
    wkv([](WkvArgs& x) { x.nent = 0; }, "wkv of nothing");
    DeltaArgs de{};
    de.M = 2, de.H = 4, de.NP = 64, de.VP = 64, de.vdim = 60, de.qdiv = 2, de.nent = de.nslots = 1;
    de.kcol = 128, de.vcol = 256, de.ld = 512, de.ldy = 240, de.rows = p, de.y = p;
    de.state = f, de.pos = ip, de.la = f, de.beta = f;
    auto delta = [&](auto edit, const char* what) {
      DeltaArgs x = de;
      edit(x);
      expect_reject(dnn_delta_steps(&x, 0, st), what);
      expect_reject(dnn_delta_chunks(&x, st), what);
    };
    delta([](DeltaArgs& x) { x.NP = 96; }, "delta key size 96");
    delta([](DeltaArgs& x) { x.vdim = 65; }, "delta head past its padding");
    delta([](DeltaArgs& x) { x.ld = 504; }, "delta row too short");
    delta([](DeltaArgs& x) { x.kcol = 448; }, "delta keys past the row");
    delta([](DeltaArgs& x) { x.ldy = 200; }, "delta result row too short");
    delta([](DeltaArgs& x) { x.beta = nullptr; }, "delta without step sizes");
    delta([](DeltaArgs& x) { x.qdiv = 0; }, "delta heads over no key heads");
    de.kcol = 132;
    expect_reject(dnn_delta_chunks(&de, st), "delta keys unaligned");
  }
  {
    RowsArgs r{};
    r.x_in = f, r.x_out = f + 64, r.M = 1, r.N = r.NP = r.ldx = r.ldh = 64, r.n_w = f, r.h = p;
    r.sh_mu = r.sh_state = f, r.sh_start = r.sh_last = r.sh_slots = r.sh_pos = ip, r.sh_nslots = 1;
    auto shift = [&](auto edit, const char* what) {
      RowsArgs x = r;
      edit(x);
      expect_reject(dnn_rows_update(&x, 0, 0, st), what);
    };
    shift([](RowsArgs& x) { x.x_out = const_cast<float*>(x.x_in); }, "rows token shift in place");
    shift([](RowsArgs& x) { x.n_w = nullptr; }, "rows token shift without a norm");
    shift([](RowsArgs& x) { x.sh_state = nullptr; }, "rows token shift without a state");
    shift([](RowsArgs& x) { x.sh_nslots = 0; }, "rows token shift of no slots");
    shift([](RowsArgs& x) { x.sh_rows = 0; }, "rows token shift in groups of none");
    QkHeadsArgs q{};
    q.qkv = q.kp = q.vp = p, q.M = 1, q.H = 2, q.G = 1, q.DK = 64, q.DV = 128, q.dim = 60, q.ldq = 320, q.ldt = q.npages = 1;
    auto heads = [&](auto edit, const char* what) {
      QkHeadsArgs x = q;
      edit(x);
      expect_reject(dnn_qk_heads(&x, 0, st), what);
    };
    heads([](QkHeadsArgs& x) { x.DK = 96; }, "qk heads of 96");
    heads([](QkHeadsArgs& x) { x.dim = 65; }, "qk heads past their padding");
    heads([](QkHeadsArgs& x) { x.ldq = 256; }, "qk heads row too short");
    heads([](QkHeadsArgs& x) { x.rope.pairs = 31; }, "qk heads with more pairs than values");
    expect_reject(dnn_xielu_f32(f, 32, 1, 64, f, st), "xielu past the row");
    expect_reject(dnn_gemm_bf16(p, 64, p, 64, p, 64, nullptr, nullptr, 0, 128, 64, 64, 6, 0, st), "xielu without constants");
    expect_reject(dnn_gemm_skinny(p, 64, nullptr, p, 64, nullptr, p, 64, nullptr, nullptr, 0, 4, 64, 64, 6, 0, 0, st),
                  "skinny xielu without constants");
  }
  {
    RopeTable rt{nullptr, 4, 1.f};
    expect_reject(dnn_rope_rows(p, 64, 64, 1, 2, 64, ip, &rt, 0, st), "rope past the row");
    rt.pairs = 33;
    expect_reject(dnn_rope_rows(p, 64, 64, 1, 1, 64, ip, &rt, 0, st), "rope more pairs than columns");
    LatentPrepArgs a{};
    a.M = 1, a.QP = a.RP = 64, a.CP = 128, a.ld = 256, a.QN = 64, a.CN = 129, a.rope.pairs = 4, a.ldt = a.npages = 1;
    expect_reject(dnn_latent_prep(&a, 0, st), "latent norm past its padding");
    a.CN = 128, a.ld = 192;
    expect_reject(dnn_latent_prep(&a, 0, st), "latent row too short");
    LatentAttnArgs b{};
    b.M = b.H = 1, b.CP = 128, b.RP = b.hs = 64, b.ldql = b.ldo = 128, b.ldqr = 64, b.ldt = b.npages = 1, b.scale = 1.f;
    b.table = b.slots = b.pos = ip;
    auto latent = [&](auto edit, const char* what) {
      LatentAttnArgs x = b;
      edit(x);
      expect_reject(dnn_latent_attn(&x, ip, 1, 32, 1, 1, nullptr, 0, st), what);
      expect_reject(dnn_latent_attn_f32(&x, st), what);
    };
    latent([](LatentAttnArgs& x) { x.CP = 192; }, "latent size 192");
    latent([](LatentAttnArgs& x) { x.ldo = 64; }, "latent result row too short");
    latent([](LatentAttnArgs& x) { x.hs = 32; }, "latent rotated part past its head");
    latent([](LatentAttnArgs& x) { x.table = nullptr; }, "latent without a block table");
    expect_reject(dnn_latent_attn(&b, ip, 1, 48, 1, 1, nullptr, 0, st), "latent tiles of 48 rows");
    expect_reject(dnn_latent_attn(&b, ip, 1, 32, 2, 1, nullptr, 0, st), "latent splits without a workspace");
    expect_reject(dnn_latent_gather(p, 192, ip, 1, 1, ip, 0, p, 64, st), "latent gather of nothing");
    LatentKeysArgs k{};
    k.M = k.H = 1, k.keys = 64, k.DP = k.RP = k.VP = 64, k.ldq = k.ldkv = 128, k.ldr = k.ldo = 64, k.scale = 1.f, k.pos = ip;
    auto keys = [&](auto edit, const char* what) {
      LatentKeysArgs x = k;
      edit(x);
      expect_reject(dnn_latent_prefill(&x, ip, 1, st), what);
    };
    keys([](LatentKeysArgs& x) { x.DP = 96; }, "attention over keys of 96");
    keys([](LatentKeysArgs& x) { x.ldkv = 64; }, "attention over keys, key row too short");
    keys([](LatentKeysArgs& x) { x.keys = 0; }, "attention over no keys");
  }
  expect_reject(dnn_token_gate(p, 64, p, 64, p, 64, p, 24, 8, ip, 5, p, 64, 4, 24, 64, st), "token gate past the row");
  expect_reject(dnn_token_gate(p, 64, p, 64, nullptr, 64, p, 24, 0, ip, 5, p, 64, 4, 24, 64, st),
                "token gate without the fragment copy");
  expect_reject(dnn_token_gate(p, 64, p, 64, p, 64, p, 24, 0, ip, 5, p, 64, 4, 24, 48, st), "token gate np%64");
  expect_reject(dnn_gemm_f32(f, 24, f, 24, f, 8, nullptr, 4, 8, 24, st), "f32 gemm K%16");
  expect_reject(dnn_glu_f32(f, 16, f, 16, 4, 12, 3, nullptr, st), "glu F%8");
  expect_reject(dnn_glu_f32(f, 16, f, 16, 4, 8, 1, nullptr, st), "glu with a plain activation");
  PagedAttnArgs pa = {};
  pa.qkv = pa.kp = pa.vp = pa.out = p, pa.table = pa.slots = pa.pos = ip;
  pa.ldq = 256, pa.ldo = 64, pa.ldt = 1, pa.npages = 1, pa.M = 1, pa.H = pa.G = 1, pa.DK = pa.DV = 64;
  pa.gate = 192, pa.window = 8, pa.keep = 0, pa.scale = 1.f;
  auto bad = [&](auto edit, const char* what) {
    PagedAttnArgs b = pa;
    edit(b);
    expect_reject(dnn_paged_decode(&b, ip, 1, 1, nullptr, 0, st), what);
    expect_reject(dnn_paged_prefill(&b, ip, 1, st), what);
    expect_reject(dnn_paged_mixed(&b, ip, 1, ip, 1, 1, nullptr, 0, st), what);
  };
  bad([](PagedAttnArgs& b) { b.DK = 96; }, "paged head size 96");
  bad([](PagedAttnArgs& b) { b.G = 2; }, "paged heads % kv heads");
  bad([](PagedAttnArgs& b) { b.ldq = 128; }, "paged qkv row too short");
  bad([](PagedAttnArgs& b) { b.window = 0; }, "paged empty window");
  bad([](PagedAttnArgs& b) { b.gate = 256; }, "paged gate past the row");
  bad([](PagedAttnArgs& b) { b.scale = -1.f; }, "paged negative scale");
  bad([](PagedAttnArgs& b) { b.table = nullptr; }, "paged without a block table");
  bad([](PagedAttnArgs& b) { b.gate_el = 1, b.gate = 196; }, "paged gate per element past the row");
  bad([](PagedAttnArgs& b) { b.shared = 1, b.written = 0; }, "paged shared keys that nobody wrote");
  expect_reject(dnn_paged_decode(&pa, ip, 1, 2, f, 4, st), "paged decode workspace too small");
  expect_reject(dnn_paged_decode(&pa, ip, 0, 1, nullptr, 0, st), "paged decode of nothing");
  expect_reject(dnn_paged_prefill(&pa, ip, 0, st), "paged prefill of nothing");
  expect_reject(dnn_paged_mixed(&pa, ip, 0, ip, 1, 1, nullptr, 0, st), "paged launch of both without portions");
  expect_reject(dnn_paged_mixed(&pa, ip, 1, ip, 0, 1, nullptr, 0, st), "paged launch of both without single tokens");
  expect_reject(dnn_paged_mixed(&pa, ip + 1, 1, ip, 1, 1, nullptr, 0, st), "paged tiles off 16 bytes");
  expect_reject(dnn_paged_mixed(&pa, ip, 1, ip, 1, 2, f, 4, st), "paged workspace of both too small");
  expect_reject(dnn_paged_mixed(&pa, ip, 0x7fffffff, ip, 1, 1, nullptr, 0, st), "paged workgroups past an int");
  // GEMMs
  expect_reject(dnn_gemm_bf16(p, 96, p, 96, p, 8, nullptr, nullptr, 0, 128, 128, 96, 0, 0, st), "gemm K%64");
  expect_reject(dnn_gemm_bf16(p, 64, p, 64, p, 8, nullptr, nullptr, 0, 0, 128, 64, 0, 0, st), "gemm M=0");
  expect_reject(dnn_gemm_set_tile(64), "gemm tile 64");
  expect_reject(dnn_gemm_skinny(p, 64, nullptr, p, 64, nullptr, p, 8, nullptr, nullptr, 0, 257, 16, 64, 0, 0, 0, st),
                "skinny M>256");
  expect_reject(dnn_gemm_skinny(p, 64, f, p, 64, f, p, 8, nullptr, nullptr, 0, 65, 16, 64, 0, 0, 1, st),
                "skinny fp8 M>64");
  expect_reject(dnn_gemm_skinny(p, 64, nullptr, p, 64, nullptr, p, 8, nullptr, nullptr, 0, 4, 16, 64, 0, 0, 1, st),
                "skinny fp8 without scales");
  expect_reject(dnn_gemm_skinny(p, 48, nullptr, p, 48, nullptr, p, 8, nullptr, nullptr, 0, 4, 24, 48, 3, 0, 0, st),
                "skinny silu N%16");
  expect_reject(dnn_gemm_skinny_norm(p, 64, p, 64, p, 8, nullptr, nullptr, 0, 4, 16, 64, 0, 2, nullptr, 1e-5f, st),
                "skinny LN without colsum");
  expect_reject(dnn_gemm_skinny_norm(p, 64, p, 64, p, 8, nullptr, nullptr, 0, 4, 16, 64, 2, 1, nullptr, 1e-5f, st),
                "skinny norm unsupported act");
  expect_reject(dnn_gemm_skinny_w8(p, 96, p, 96, f, p, 8, nullptr, nullptr, 0, 4, 16, 96, 0, 0, nullptr, 0.f, st),
                "w8 K%64");
  expect_reject(dnn_gemm_skinny_w8(p, 64, p, 32, f, p, 8, nullptr, nullptr, 0, 4, 16, 64, 0, 0, nullptr, 0.f, st),
                "w8 ldw < K");
  expect_reject(dnn_gemm_skinny_w8(p, 64, p, 64, nullptr, p, 8, nullptr, nullptr, 0, 4, 16, 64, 0, 0, nullptr, 0.f,
                                   st), "w8 without scales");
  expect_reject(dnn_gemm_skinny_sweep(p, 64, p, 64, nullptr, p, 8, 4, 16, 64, 1, 2, 16, 0, 0, st), "sweep ks>8");
  expect_reject(dnn_gemm_fp8(p, f, p, f, p, 8, nullptr, nullptr, 0, 128, 128, 96, 0, st), "fp8 K%128");
  expect_reject(dnn_gemm_fp8(p, f, p, f, p, 8, nullptr, nullptr, 0, 128, 24, 128, 3, st), "fp8 silu N%16");
  const int wide = 1 << 29;  // 7 rows of it are the 32-bit row offsets of the 256 x 256 tiles
  expect_reject(dnn_gemm_fp8_256(p, f, p, f, p, 256, nullptr, nullptr, 0, 256, 256, wide, 0, st), "fp8 256 x 256 wide rows");
  expect_reject(dnn_gemm_fp8_mx(p, p, p, f, p, 256, nullptr, nullptr, 0, 256, 256, wide, 0, nullptr, 0, nullptr, 0, st),
                "MX wide rows");
  expect_reject(dnn_gemm_fp8_qkv_scatter(p, f, p, f, nullptr, p, p, p, ip, 1, 256, 2, 1, 64, 256, wide, st),
                "fp8 scatter wide rows");
  expect_reject(dnn_gemm_fp8_qkv_scatter_mx(p, p, p, f, nullptr, p, p, p, ip, 1, 256, 2, 1, 64, 256, wide, st),
                "MX scatter wide rows");
  expect_reject(dnn_quant_fp8_rows(p, 12, p, f, 4, 12, 128, st), "quant K%8");
  expect_reject(dnn_quant_fp8_rows(p, 256, p, f, 4, 256, 128, st), "quant kpad<K");
  // norms / embedding
  expect_reject(dnn_layernorm(p, 12, f, f, p, 12, 4, 12, 1e-5f, 0, st), "layernorm N%8");
  expect_reject(dnn_layernorm(p, 16384, f, f, p, 16384, 4, 16384, 1e-5f, 1, st), "layernorm N>8192");
  expect_reject(dnn_embed_gpt2(ip, p, p, p, 1, 1, 12, ip, 8, 8, st), "embed d%8");
  expect_reject(dnn_embed_gpt2(ip, p, p, p, 1, 1, 16, ip, 0, 8, st), "embed empty vocab");
  expect_reject(dnn_layernorm_q8_mx(p, 64, nullptr, f, p, 128, p, 4, 64, 128, 1e-5f, 0, st), "standardised rows with a shift");
  expect_reject(dnn_layernorm_q8_mx(p, 68, nullptr, nullptr, p, 128, p, 4, 64, 128, 1e-5f, 0, st), "standardised rows ld%8");
  expect_reject(dnn_layernorm_q8_mx(buf + 8, 64, nullptr, nullptr, p, 128, p, 4, 64, 128, 1e-5f, 0, st),
                "standardised rows off 16 bytes");
  // attention
  auto rope = [&](int K, int hd, int T, const float* table) {
    return dnn_gemm_bf16_qkv_rope(p, K, p, K, 1e-5f, f, p, p, p, ip, 1, T, 2, 1, hd, 512, K, table, table, 0, st);
  };
  expect_eq(rope(96, 128, 300, f), -3, "rotating projection K%64");
  expect_eq(rope(128, 64, 300, f), -3, "rotating projection hd=64");
  expect_eq(rope(128, 128, 300, f + 1), -3, "rotating projection tables off 16 bytes");
  expect_eq(rope(128, 128, 0, f), -1, "rotating projection of nothing");
  expect_eq(rope(128, 128, 300, nullptr), -1, "rotating projection without tables");
  auto mx = [&](int T, int H, int Hkv, int hd, int ld8) {
    return dnn_flash_attn_mx(p, p, p, p, ld8, p, 1, T, H, Hkv, hd, T, ip, 0.1f, st);
  };
  expect_eq(mx(64, 6, 4, 64, 384), -1, "flash that quantises H%Hkv");
  expect_eq(mx(64, 5, 5, 64, 320), -1, "flash that quantises, row too short");
  expect_eq(mx(64, 4, 4, 128, 512), -3, "flash that quantises hd=128");
  expect_eq(mx(2048, 4, 4, 64, 256), -3, "flash that quantises, long");
  const RowBlock block = {p, p, p, p, f, f, f, f, f, f};
  auto row = [&](int n, int M, int d, int H, int hd, int S) {
    return dnn_decode_row_blocks(&block, n, p, p, p, p, p, f, buf, buf, 0, M, d, H, H, hd, S, ip, 0.1f, 1e-5f, st);
  };
  expect_eq(row(0, 1, 768, 12, 64, 64), -3, "row step without blocks");
  expect_eq(row(1, 3, 768, 12, 64, 64), -3, "row step of three rows");
  expect_eq(row(1, 1, 1280, 20, 64, 64), -3, "row step width 1280");
  expect_eq(row(1, 1, 768, 6, 128, 64), -3, "row step hd=128");
  expect_eq(row(1, 1, 768, 12, 64, 2048), -3, "row step of a split cache");
  expect_reject(dnn_attn_decode_proj(p, 2304, p, p, p, f, 0, 12, 64, ip, 0.1f, st), "attention and projection of nothing");
  expect_reject(dnn_attn_decode_proj(p, 2296, p, p, p, f, 1, 12, 64, ip, 0.1f, st), "attention and projection, row too short");
  expect_reject(dnn_attn_decode_proj(p, 2308, p, p, p, f, 1, 12, 64, ip, 0.1f, st), "attention and projection ld%8");
  expect_reject(dnn_qkv_split(p, p, p, p, 1, 1, 4, 4, 24, 16, ip, nullptr, nullptr, 0, st), "qkv_split hd%16");
  expect_reject(dnn_qkv_split(p, p, p, p, 1, 1, 6, 4, 64, 16, ip, nullptr, nullptr, 0, st), "qkv_split H%Hkv");
  expect_reject(dnn_flash_attn(p, p, p, p, 1, 8, 6, 4, 64, 16, ip, 0.1f, st), "flash H%Hkv");
  expect_reject(dnn_flash_attn(p, p, p, p, 1, 8, 4, 4, 96, 16, ip, 0.1f, st), "flash hd=96");
  expect_reject(dnn_attn_decode(p, p, p, p, 1, 4, 4, 64, 16, ip, 0.1f, 0, f, st), "decode splits=0");
  expect_reject(dnn_attn_decode(p, p, p, p, 1, 32, 2, 64, 16, ip, 0.1f, 1, f, st), "decode G>8");
  expect_reject(dnn_attn_decode(p, p, p, p, 1, 4, 4, 96, 16, ip, 0.1f, 1, f, st), "decode hd=96");
  expect_reject(dnn_attn_decode(p, p, p, p, 1, 8, 2, 64, 16, ip, 0.1f, 1, f, st, 1), "decode fp8 KV, GQA at hd 64");
  expect_reject(dnn_attn_decode_qkv(p, 100, p, p, p, 1, 4, 4, 64, 16, ip, nullptr, nullptr, 0.1f, 1, f, st),
                "decode_qkv ldqkv too small");
  // sampling
  expect_reject(dnn_sample_topk(p, 16, 2, 16, ip, 0.f, 0, 1u, nullptr, st), "sample temperature 0");
  expect_reject(dnn_sample_topk(p, 12, 2, 12, ip, 1.f, 0, 1u, nullptr, st), "sample ld%8");
  expect_reject(dnn_argmax_rows(p, 12, 2, 12, ip, 0, st), "argmax bf16 ld%8");
  expect_noop(dnn_argmax_rows(p, 16, 0, 16, ip, 0, st), "argmax M=0");
  // CIFAR
  expect_reject(dnn_cifar_set_v4_pt(3), "v4 pt%4");
  expect_reject(dnn_cifar_set_v4_pt(36), "v4 pt>32");
  expect_noop(dnn_cifar_stage0_v4(f, p, p, f, p, f, 0, 0, st), "stage0 B=0");
  expect_noop(dnn_cifar_head_tail(p, p, f, f, ip, 0, st), "head B=0");
  for (int off = 0; off < 3; ++off) {  // rows or weights that 16-byte LDS-DMA does not fetch
    char* q[3] = {buf, buf, buf};
    q[off] += 4;
    expect_reject(dnn_cifar_fc1_x3(reinterpret_cast<float*>(q[0]), 4096, q[1], q[2], 4096, f, f, 512, 600, 512, 4096, st),
                  "fc1 operands off 16 bytes");
  }
  expect_eq(dnn_cifar_fc1_ranges(16384, 512, 2, f, f, f), 2, "fc1 ranges");
  expect_eq(dnn_cifar_fc1_ranges(1 << 22, 2048, 2, f, f, f), 1, "fc1 ranges of 2^31 quads of columns");
  expect_eq(dnn_cifar_fc1_ranges(1 << 20, 4096, 2, f, f, f), 2, "fc1 ranges of 2^30 quads of columns");
  expect_eq(dnn_cifar_fc1_ranges(600, 512, 2, f + 1, f, f), 1, "fc1 ranges into rows off 16 bytes");
  if (g_fail) {
    std::printf("host_validate FAILED (%d)\n", g_fail);
    return 1;
  }
  std::printf("host_validate ok\n");
  return 0;
}
