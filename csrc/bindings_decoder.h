// Bindings shared by the full kernel library (bindings.cpp) and the decoder
// subset (bindings_decoder.cpp): the bf16 / fp32 GEMMs, the sampler, and the
// fp32-residual and paged-attention kernels.
#pragma once
#include <pybind11/pybind11.h>
#include <pybind11/stl.h>
#include <hip/hip_runtime.h>
#include <cstdint>

#include "kernels/api.h"
#include "kernels/mixer_api.h"
#include "kernels/residual_api.h"

namespace py = pybind11;
#define P(x) reinterpret_cast<void*>(static_cast<uintptr_t>(x))
#define CP(x) reinterpret_cast<const void*>(static_cast<uintptr_t>(x))
#define FP(x) reinterpret_cast<float*>(static_cast<uintptr_t>(x))
#define CFP(x) reinterpret_cast<const float*>(static_cast<uintptr_t>(x))
#define IP(x) reinterpret_cast<int*>(static_cast<uintptr_t>(x))
#define CIP(x) reinterpret_cast<const int*>(static_cast<uintptr_t>(x))
#define ST(x) reinterpret_cast<hipStream_t>(static_cast<uintptr_t>(x))
typedef uint64_t u64;

inline void bind_decoder(py::module_& m) {
  m.def("gemm_bf16", [](u64 A, int lda, u64 W, int ldw, u64 C, int ldc, u64 bias, u64 R, int ldr, int M, int N,
                        int K, int act, int out_f32, u64 st, u64 wsh, u64 rowstat, u64 colsum, u64 ws,
                        long long ws_bytes) {
    return dnn_gemm_bf16(CP(A), lda, CP(W), ldw, P(C), ldc, CFP(bias), CP(R), ldr, M, N, K, act, out_f32, ST(st),
                         CP(wsh), CFP(rowstat), CFP(colsum), P(ws), ws_bytes);
  }, py::arg("A"), py::arg("lda"), py::arg("W"), py::arg("ldw"), py::arg("C"), py::arg("ldc"), py::arg("bias"),
     py::arg("R"), py::arg("ldr"), py::arg("M"), py::arg("N"), py::arg("K"), py::arg("act"), py::arg("out_f32"),
     py::arg("st"), py::arg("wsh") = 0, py::arg("rowstat") = 0, py::arg("colsum") = 0, py::arg("ws") = 0,
     py::arg("ws_bytes") = 0);
  m.def("gemm_set_mid", [](int tile, int splits) { return dnn_gemm_set_mid(tile, splits); });
  m.def("gemm_mid_blocks", [](int tile, int mx) { return dnn_gemm_mid_blocks(tile, mx); });
  m.def("gemm_is_skinny", [](int M, int N, int K, int norm, int frag, long long ws_bytes) {
    return dnn_gemm_is_skinny(M, N, K, norm, frag, ws_bytes);
  });
  m.def("sample_topk", [](u64 x, int ld, int M, int N, u64 out, float temperature, int topk, unsigned seed, u64 step,
                          u64 st) {
    return dnn_sample_topk(CP(x), ld, M, N, reinterpret_cast<int*>(out), temperature, topk, seed,
                           reinterpret_cast<const int*>(step), ST(st));
  });
  m.def("argmax_rows", [](u64 x, int ld, int M, int N, u64 out, int f32in, u64 st, u64 out2, u64 pos_inc, u64 part,
                          u64 hist, int hist_ld) {
    return dnn_argmax_rows(CP(x), ld, M, N, IP(out), f32in, ST(st), IP(out2), IP(pos_inc),
                           reinterpret_cast<void*>(static_cast<uintptr_t>(part)), IP(hist), hist_ld);
  }, py::arg("x"), py::arg("ld"), py::arg("M"), py::arg("N"), py::arg("out"), py::arg("f32in"), py::arg("st"),
     py::arg("out2") = 0, py::arg("pos_inc") = 0, py::arg("part") = 0, py::arg("hist") = 0, py::arg("hist_ld") = 0);
  // argument structs: pointers as addresses, every field by name
#define PF(S, f) .def_property(#f, [](const S& a) { return (u64)(uintptr_t)a.f; }, [](S& a, u64 v) { a.f = reinterpret_cast<decltype(a.f)>(static_cast<uintptr_t>(v)); })
#define VF(S, f) .def_readwrite(#f, &S::f)
  py::class_<RowsArgs>(m, "RowsArgs")
      .def(py::init([] { return RowsArgs{}; }))
      PF(RowsArgs, x_in) PF(RowsArgs, xidx) PF(RowsArgs, y) PF(RowsArgs, yidx) PF(RowsArgs, y_w) PF(RowsArgs, x_out)
      PF(RowsArgs, copy) PF(RowsArgs, n_w) PF(RowsArgs, h) PF(RowsArgs, x_add) PF(RowsArgs, y2) PF(RowsArgs, y2_w)
      PF(RowsArgs, ys) PF(RowsArgs, ysi) PF(RowsArgs, ysw) PF(RowsArgs, n_b) PF(RowsArgs, pos) PF(RowsArgs, freq)
      VF(RowsArgs, xrows) VF(RowsArgs, yrows) VF(RowsArgs, ldx) VF(RowsArgs, ldy) VF(RowsArgs, ldcopy) VF(RowsArgs, ldh)
      VF(RowsArgs, M) VF(RowsArgs, N) VF(RowsArgs, NP) VF(RowsArgs, mult) VF(RowsArgs, eps) VF(RowsArgs, ldadd)
      VF(RowsArgs, ldy2) VF(RowsArgs, ldys) VF(RowsArgs, ysrows) VF(RowsArgs, top) VF(RowsArgs, n_alpha) VF(RowsArgs, y_joined)
      PF(RowsArgs, sh_mu) PF(RowsArgs, sh_state) PF(RowsArgs, sh_start) PF(RowsArgs, sh_last) PF(RowsArgs, sh_slots)
      PF(RowsArgs, sh_pos) VF(RowsArgs, sh_nslots) VF(RowsArgs, sh_rows);
  m.def("rows_update", [](const RowsArgs& a, int y_f32, int out_f32, u64 st) {
    return dnn_rows_update(&a, y_f32, out_f32, ST(st));
  });
  py::class_<QkNormArgs>(m, "QkNormArgs")
      .def(py::init([] { return QkNormArgs{}; }))
      PF(QkNormArgs, qkv) PF(QkNormArgs, kp) PF(QkNormArgs, kscale) PF(QkNormArgs, qw) PF(QkNormArgs, table)
      PF(QkNormArgs, slots) PF(QkNormArgs, pos) VF(QkNormArgs, ldq) VF(QkNormArgs, ldt) VF(QkNormArgs, npages)
      VF(QkNormArgs, M) VF(QkNormArgs, H) VF(QkNormArgs, G) VF(QkNormArgs, DK) VF(QkNormArgs, nq) VF(QkNormArgs, nk)
      VF(QkNormArgs, t_every) VF(QkNormArgs, t_coef) VF(QkNormArgs, eps);
  m.def("qk_norm", [](const QkNormArgs& a, int f32, u64 st) { return dnn_qk_norm(&a, f32, ST(st)); });
  py::class_<ConvArgs>(m, "ConvArgs")
      .def(py::init([] { return ConvArgs{}; }))
      PF(ConvArgs, in) PF(ConvArgs, w) PF(ConvArgs, b) PF(ConvArgs, ring) PF(ConvArgs, out) PF(ConvArgs, start)
      PF(ConvArgs, slots) PF(ConvArgs, pos) PF(ConvArgs, dt_bias) PF(ConvArgs, a_log) PF(ConvArgs, dt) PF(ConvArgs, la)
      VF(ConvArgs, ldi) VF(ConvArgs, ldo) VF(ConvArgs, M) VF(ConvArgs, C) VF(ConvArgs, taps) VF(ConvArgs, dt_col)
      VF(ConvArgs, H) VF(ConvArgs, nslots) VF(ConvArgs, b_col);
  m.def("conv", [](const ConvArgs& a, int f32, u64 st) { return dnn_conv(&a, f32, ST(st)); });
  m.def("conv_state", [](const ConvArgs& a, u64 ent, int nent, int f32, u64 st) {
    return dnn_conv_state(&a, reinterpret_cast<const int4*>(CP(ent)), nent, f32, ST(st));
  });
  py::class_<ScanArgs>(m, "ScanArgs")
      .def(py::init([] { return ScanArgs{}; }))
      PF(ScanArgs, rows) PF(ScanArgs, dt) PF(ScanArgs, la) PF(ScanArgs, la_h) PF(ScanArgs, D) PF(ScanArgs, state)
      PF(ScanArgs, y) PF(ScanArgs, ent) PF(ScanArgs, pos) VF(ScanArgs, ld) VF(ScanArgs, ldy) VF(ScanArgs, qcol)
      VF(ScanArgs, kcol) VF(ScanArgs, vcol) VF(ScanArgs, qdiv) VF(ScanArgs, M) VF(ScanArgs, H) VF(ScanArgs, NP)
      VF(ScanArgs, VP) VF(ScanArgs, vdim) VF(ScanArgs, nent) VF(ScanArgs, nslots) VF(ScanArgs, dt_c);
  m.def("scan_steps", [](const ScanArgs& a, int f32, u64 st) { return dnn_scan_steps(&a, f32, ST(st)); });
  m.def("scan_chunks", [](const ScanArgs& a, u64 st) { return dnn_scan_chunks(&a, ST(st)); });
  py::class_<DeltaArgs>(m, "DeltaArgs")
      .def(py::init([] { return DeltaArgs{}; }))
      PF(DeltaArgs, rows) PF(DeltaArgs, beta) PF(DeltaArgs, la) PF(DeltaArgs, state) PF(DeltaArgs, y) PF(DeltaArgs, ent)
      PF(DeltaArgs, pos) VF(DeltaArgs, ld) VF(DeltaArgs, ldy) VF(DeltaArgs, qcol) VF(DeltaArgs, kcol) VF(DeltaArgs, vcol)
      VF(DeltaArgs, qdiv) VF(DeltaArgs, M) VF(DeltaArgs, H) VF(DeltaArgs, NP) VF(DeltaArgs, VP) VF(DeltaArgs, vdim)
      VF(DeltaArgs, nent) VF(DeltaArgs, nslots) VF(DeltaArgs, q_scale) VF(DeltaArgs, unit_eps);
  m.def("delta_steps", [](const DeltaArgs& a, int f32, u64 st) { return dnn_delta_steps(&a, f32, ST(st)); });
  m.def("delta_chunks", [](const DeltaArgs& a, u64 st) { return dnn_delta_chunks(&a, ST(st)); });
  py::class_<PairArgs>(m, "PairArgs")
      .def(py::init([] { return PairArgs{}; }))
      PF(PairArgs, ids) PF(PairArgs, start) PF(PairArgs, last) PF(PairArgs, slots) PF(PairArgs, pos) PF(PairArgs, prev)
      PF(PairArgs, rows) VF(PairArgs, mul_prev) VF(PairArgs, mul_cur) VF(PairArgs, buckets) VF(PairArgs, M)
      VF(PairArgs, nslots);
  m.def("pair_rows", [](const PairArgs& a, u64 st) { return dnn_pair_rows(&a, ST(st)); });
  py::class_<ShiftArgs>(m, "ShiftArgs")
      .def(py::init([] { return ShiftArgs{}; }))
      PF(ShiftArgs, x) PF(ShiftArgs, mu) PF(ShiftArgs, out) PF(ShiftArgs, state) PF(ShiftArgs, start) PF(ShiftArgs, last)
      PF(ShiftArgs, slots) PF(ShiftArgs, pos) VF(ShiftArgs, ostride) VF(ShiftArgs, ldx) VF(ShiftArgs, ldo) VF(ShiftArgs, M)
      VF(ShiftArgs, NP) VF(ShiftArgs, n) VF(ShiftArgs, nslots);
  m.def("token_shift", [](const ShiftArgs& a, int f32, u64 st) { return dnn_token_shift(&a, f32, ST(st)); });
  py::class_<DecayArgs>(m, "DecayArgs")
      .def(py::init([] { return DecayArgs{}; }))
      PF(DecayArgs, t) PF(DecayArgs, w2) PF(DecayArgs, w0) PF(DecayArgs, la) VF(DecayArgs, ldt) VF(DecayArgs, M)
      VF(DecayArgs, N) VF(DecayArgs, rank);
  m.def("decay", [](const DecayArgs& a, int f32, u64 st) { return dnn_decay(&a, f32, ST(st)); });
  py::class_<WkvArgs>(m, "WkvArgs")
      .def(py::init([] { return WkvArgs{}; }))
      PF(WkvArgs, r) PF(WkvArgs, k) PF(WkvArgs, v) PF(WkvArgs, la) PF(WkvArgs, u) PF(WkvArgs, state) PF(WkvArgs, y)
      PF(WkvArgs, ent) PF(WkvArgs, pos) VF(WkvArgs, ld) VF(WkvArgs, ldy) VF(WkvArgs, M) VF(WkvArgs, H) VF(WkvArgs, NP)
      VF(WkvArgs, dim) VF(WkvArgs, nent) VF(WkvArgs, nslots);
  m.def("wkv_steps", [](const WkvArgs& a, int f32, u64 st) { return dnn_wkv_steps(&a, f32, ST(st)); });
  m.def("wkv_chunks", [](const WkvArgs& a, u64 st) { return dnn_wkv_chunks(&a, ST(st)); });
  py::class_<PolyNormArgs>(m, "PolyNormArgs")
      .def(py::init([] { return PolyNormArgs{}; }))
      PF(PolyNormArgs, z) PF(PolyNormArgs, w) VF(PolyNormArgs, ld) VF(PolyNormArgs, M) VF(PolyNormArgs, n)
      VF(PolyNormArgs, eps);
  m.def("poly_norm", [](const PolyNormArgs& a, int f32, u64 st) { return dnn_poly_norm(&a, f32, ST(st)); });
  py::class_<RopeTable>(m, "RopeTable")
      .def(py::init([](u64 freq, int pairs, float mag) {
        RopeTable r;
        r.freq = reinterpret_cast<const double*>(CP(freq)), r.pairs = pairs, r.mag = mag;
        return r;
      }));
  py::class_<QkHeadsArgs>(m, "QkHeadsArgs")
      .def(py::init([] { return QkHeadsArgs{}; }))
      PF(QkHeadsArgs, qkv) PF(QkHeadsArgs, kp) PF(QkHeadsArgs, vp) PF(QkHeadsArgs, table) PF(QkHeadsArgs, slots)
      PF(QkHeadsArgs, pos) VF(QkHeadsArgs, rope) VF(QkHeadsArgs, ldq) VF(QkHeadsArgs, ldt) VF(QkHeadsArgs, npages)
      VF(QkHeadsArgs, M) VF(QkHeadsArgs, H) VF(QkHeadsArgs, G) VF(QkHeadsArgs, DK) VF(QkHeadsArgs, DV)
      VF(QkHeadsArgs, dim) VF(QkHeadsArgs, eps);
  m.def("qk_heads", [](const QkHeadsArgs& a, int f32, u64 st) { return dnn_qk_heads(&a, f32, ST(st)); });
  m.def("xielu_f32", [](u64 z, int ld, int M, int n, u64 c, u64 st) { return dnn_xielu_f32(FP(z), ld, M, n, CFP(c), ST(st)); });
  m.def("rope_rows", [](u64 x, int ld, int hs, int M, int H, int RP, u64 pos, const RopeTable& r, int f32, u64 st) {
    return dnn_rope_rows(P(x), ld, hs, M, H, RP, CIP(pos), &r, f32, ST(st));
  });
  py::class_<LatentPrepArgs>(m, "LatentPrepArgs")
      .def(py::init([] { return LatentPrepArgs{}; }))
      PF(LatentPrepArgs, rows) PF(LatentPrepArgs, kp) PF(LatentPrepArgs, qw) PF(LatentPrepArgs, cw)
      PF(LatentPrepArgs, table) PF(LatentPrepArgs, slots) PF(LatentPrepArgs, pos) VF(LatentPrepArgs, rope)
      VF(LatentPrepArgs, ld) VF(LatentPrepArgs, ldt) VF(LatentPrepArgs, npages) VF(LatentPrepArgs, M)
      VF(LatentPrepArgs, QN) VF(LatentPrepArgs, QP) VF(LatentPrepArgs, CN) VF(LatentPrepArgs, CP) VF(LatentPrepArgs, RP)
      VF(LatentPrepArgs, eps);
  m.def("latent_prep", [](const LatentPrepArgs& a, int f32, u64 st) { return dnn_latent_prep(&a, f32, ST(st)); });
  py::class_<LatentAttnArgs>(m, "LatentAttnArgs")
      .def(py::init([] { return LatentAttnArgs{}; }))
      PF(LatentAttnArgs, qlat) PF(LatentAttnArgs, qrot) PF(LatentAttnArgs, kp) PF(LatentAttnArgs, table)
      PF(LatentAttnArgs, slots) PF(LatentAttnArgs, pos) PF(LatentAttnArgs, out) PF(LatentAttnArgs, gate)
      VF(LatentAttnArgs, ldql) VF(LatentAttnArgs, ldqr) VF(LatentAttnArgs, hs) VF(LatentAttnArgs, ldo)
      VF(LatentAttnArgs, ldg) VF(LatentAttnArgs, ldt) VF(LatentAttnArgs, npages) VF(LatentAttnArgs, M)
      VF(LatentAttnArgs, H) VF(LatentAttnArgs, CP) VF(LatentAttnArgs, RP) VF(LatentAttnArgs, scale);
  m.def("latent_attn", [](const LatentAttnArgs& a, u64 tiles, int ntiles, int rows, int splits, int per_token, u64 ws,
                          long long ws_elems, u64 st) {
    return dnn_latent_attn(&a, CIP(tiles), ntiles, rows, splits, per_token, FP(ws), ws_elems, ST(st));
  });
  m.def("latent_gather", [](u64 kp, int cols, u64 table, int ldt, int npages, u64 ent, int nent, u64 out, int rows, u64 st) {
    return dnn_latent_gather(P(kp), cols, CIP(table), ldt, npages, CIP(ent), nent, P(out), rows, ST(st));
  });
  py::class_<LatentKeysArgs>(m, "LatentKeysArgs")
      .def(py::init([] { return LatentKeysArgs{}; }))
      PF(LatentKeysArgs, q) PF(LatentKeysArgs, kv) PF(LatentKeysArgs, krot) PF(LatentKeysArgs, pos) PF(LatentKeysArgs, out)
      PF(LatentKeysArgs, gate) VF(LatentKeysArgs, ldq) VF(LatentKeysArgs, ldkv) VF(LatentKeysArgs, ldr)
      VF(LatentKeysArgs, ldo) VF(LatentKeysArgs, ldg) VF(LatentKeysArgs, M) VF(LatentKeysArgs, H) VF(LatentKeysArgs, DP)
      VF(LatentKeysArgs, RP) VF(LatentKeysArgs, VP) VF(LatentKeysArgs, keys) VF(LatentKeysArgs, scale);
  m.def("latent_prefill", [](const LatentKeysArgs& a, u64 tiles, int ntiles, u64 st) {
    return dnn_latent_prefill(&a, CIP(tiles), ntiles, ST(st));
  });
  m.def("latent_attn_f32", [](const LatentAttnArgs& a, u64 st) { return dnn_latent_attn_f32(&a, ST(st)); });
  py::class_<GatedNormArgs>(m, "GatedNormArgs")
      .def(py::init([] { return GatedNormArgs{}; }))
      PF(GatedNormArgs, y) PF(GatedNormArgs, z) PF(GatedNormArgs, w) PF(GatedNormArgs, out) VF(GatedNormArgs, ldy)
      VF(GatedNormArgs, ldz) VF(GatedNormArgs, ldo) VF(GatedNormArgs, M) VF(GatedNormArgs, n) VF(GatedNormArgs, groups)
      VF(GatedNormArgs, gate_first) VF(GatedNormArgs, eps);
  m.def("gated_norm", [](const GatedNormArgs& a, int f32, u64 st) { return dnn_gated_norm(&a, f32, ST(st)); });
  py::class_<RouteArgs>(m, "RouteArgs")
      .def(py::init([] { return RouteArgs{}; }))
      PF(RouteArgs, logits) PF(RouteArgs, idx) PF(RouteArgs, w) PF(RouteArgs, rank) PF(RouteArgs, counts)
      PF(RouteArgs, order) PF(RouteArgs, place) PF(RouteArgs, offs) VF(RouteArgs, ldl) VF(RouteArgs, M) VF(RouteArgs, E)
      VF(RouteArgs, groups) VF(RouteArgs, keep) VF(RouteArgs, top) PF(RouteArgs, correction) VF(RouteArgs, sigmoid) VF(RouteArgs, group_top)
      VF(RouteArgs, normalise);
  m.def("route", [](const RouteArgs& a, u64 st) { return dnn_route(&a, ST(st)); });
  py::class_<GroupedArgs>(m, "GroupedArgs")
      .def(py::init([] { return GroupedArgs{}; }))
      PF(GroupedArgs, A) PF(GroupedArgs, W) PF(GroupedArgs, Wsh) PF(GroupedArgs, C) PF(GroupedArgs, offs)
      PF(GroupedArgs, order) PF(GroupedArgs, counts) VF(GroupedArgs, lda) VF(GroupedArgs, ldc) VF(GroupedArgs, rows)
      VF(GroupedArgs, arows) VF(GroupedArgs, div) VF(GroupedArgs, N) VF(GroupedArgs, K) VF(GroupedArgs, E)
      VF(GroupedArgs, act) VF(GroupedArgs, sa) VF(GroupedArgs, sc)
      .def("set_clamp", [](GroupedArgs& a, float limit, float alpha, float shift) { a.clamp = {limit, alpha, shift}; });
  m.def("grouped_gemm", [](const GroupedArgs& a, u64 st) { return dnn_grouped_gemm(&a, ST(st)); });
  m.def("grouped_gemm_f32", [](const GroupedArgs& a, u64 st) { return dnn_grouped_gemm_f32(&a, ST(st)); });
  m.def("token_gate", [](u64 x, int ldx, u64 w, int ldw, u64 wsh, int K, u64 table, int ldt, int off, u64 tok, int V,
                         u64 g, int ldg, int M, int n, int np, u64 st) {
    return dnn_token_gate(CP(x), ldx, CP(w), ldw, CP(wsh), K, CP(table), ldt, off, CIP(tok), V, P(g), ldg, M, n, np,
                          ST(st));
  });
  m.def("token_gate_f32", [](u64 z, int ldz, u64 table, int ldt, int off, u64 tok, int V, u64 g, int ldg, int M, int n,
                             int np, u64 st) {
    return dnn_token_gate_f32(CFP(z), ldz, CFP(table), ldt, off, CIP(tok), V, FP(g), ldg, M, n, np, ST(st));
  });
  m.def("glu_f32", [](u64 gu, int ldi, u64 out, int ldo, int M, int F, int act, u64 st, float limit, float alpha,
                      float shift) {
    const GluClamp c{limit, alpha, shift};
    return dnn_glu_f32(CFP(gu), ldi, FP(out), ldo, M, F, act, &c, ST(st));
  }, py::arg("gu"), py::arg("ldi"), py::arg("out"), py::arg("ldo"), py::arg("M"), py::arg("F"), py::arg("act"),
     py::arg("st"), py::arg("limit") = 0.f, py::arg("alpha") = 0.f, py::arg("shift") = 0.f);
  m.def("gemm_f32", [](u64 A, int lda, u64 W, int ldw, u64 C, int ldc, u64 bias, int M, int N, int K, u64 st) {
    return dnn_gemm_f32(CFP(A), lda, CFP(W), ldw, FP(C), ldc, CFP(bias), M, N, K, ST(st));
  });
  py::class_<PagedAttnArgs>(m, "PagedAttnArgs")
      .def(py::init([](u64 qkv, int ldq, u64 kp, u64 vp, u64 table, int ldt, int npages, u64 slots, u64 pos, u64 out,
                       int ldo, int M, int H, int G, int DK, int DV, int gate, int window, int keep, float scale) {
        PagedAttnArgs a;
        a.qkv = CP(qkv), a.kp = P(kp), a.vp = P(vp), a.table = CIP(table), a.slots = CIP(slots), a.pos = CIP(pos);
        a.out = P(out), a.ldq = ldq, a.ldo = ldo, a.ldt = ldt, a.npages = npages, a.M = M, a.H = H, a.G = G;
        a.DK = DK, a.DV = DV, a.gate = gate, a.window = window, a.keep = keep, a.scale = scale;
        return a;
      }))
      PF(PagedAttnArgs, kscale) PF(PagedAttnArgs, slopes) VF(PagedAttnArgs, gate_el) VF(PagedAttnArgs, shared)
      VF(PagedAttnArgs, written) PF(PagedAttnArgs, sinks);
  m.def("paged_write", [](const PagedAttnArgs& a, int f32, u64 st) { return dnn_paged_write(&a, f32, ST(st)); });
  m.def("paged_prefill", [](const PagedAttnArgs& a, u64 tiles, int ntiles, u64 st) {
    return dnn_paged_prefill(&a, CIP(tiles), ntiles, ST(st));
  });
  m.def("paged_mixed", [](const PagedAttnArgs& a, u64 tiles, int ntiles, u64 rows, int nrows, int splits, u64 ws,
                          long long ws_elems, u64 st) {
    return dnn_paged_mixed(&a, CIP(tiles), ntiles, CIP(rows), nrows, splits, FP(ws), ws_elems, ST(st));
  });
  m.def("paged_decode", [](const PagedAttnArgs& a, u64 rows, int nrows, int splits, u64 ws, long long ws_elems,
                           u64 st) {
    return dnn_paged_decode(&a, CIP(rows), nrows, splits, FP(ws), ws_elems, ST(st));
  });
  m.def("paged_attn_f32", [](const PagedAttnArgs& a, u64 st) { return dnn_paged_attn_f32(&a, ST(st)); });
}
