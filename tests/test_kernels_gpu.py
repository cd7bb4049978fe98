"""HIP kernel numerics vs plain PyTorch fp32 references (MI355X only)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _rel(a, b):
    return ((a.float() - b.float()).norm() / (b.float().norm() + 1e-12)).item()


@pytest.mark.parametrize("M,N,K", [(128, 128, 64), (256, 384, 768), (77, 200, 128), (4096, 512, 4096),
                                   (1, 768, 768), (7, 3072, 768), (16, 50257, 768), (300, 2304, 768),
                                   (32, 4096, 14336), (64, 2304, 768), (40, 100, 128), (2, 28672, 4096),
                                   (128, 768, 768), (200, 2304, 768), (256, 3072, 768), (97, 768, 3072)])
@pytest.mark.parametrize("act", [0, 1, 2])
def test_gemm_bf16(M, N, K, act):
    from distributed_neural_networks_amd.ops.gemm import linear
    torch.manual_seed(0)
    x = torch.randn(M, K, device=DEV).bfloat16()
    w = (torch.randn(N, K, device=DEV) * 0.05).bfloat16()
    b = torch.randn(N, device=DEV)
    r = torch.randn(M, N, device=DEV).bfloat16()
    y = linear(x, w, b, act=act, residual=r)
    ref = x.float() @ w.float().t() + b
    if act == 1:
        ref = torch.relu(ref)
    elif act == 2:
        ref = torch.nn.functional.gelu(ref)
    ref = ref + r.float()
    assert _rel(y, ref) < 1e-2


@pytest.mark.parametrize("M,N,K", [(256, 256, 64), (512, 512, 4096), (300, 2304, 768), (1000, 520, 192),
                                   (2048, 768, 3072), (65, 300, 128)])
@pytest.mark.parametrize("act", [0, 1, 2, 3])
@pytest.mark.parametrize("tile", [256, 255])
def test_gemm_bf16_256_tile(M, N, K, act, tile):
    """The 256x256 4-phase GEMM and its 256x128 2-phase variant (tile 255),
    forced, including edge tiles and odd K-tile counts."""
    from distributed_neural_networks_amd.ops.gemm import linear, set_gemm_tile
    if act == 3 and N % 16:
        pytest.skip("packed gate|up needs N % 16 == 0")
    torch.manual_seed(2)
    x = torch.randn(M, K, device=DEV).bfloat16()
    w = (torch.randn(N, K, device=DEV) * 0.05).bfloat16()
    b = torch.randn(N, device=DEV)
    set_gemm_tile(tile)
    try:
        if act == 3:
            y = linear(x, w, act="silu_mul")
        else:
            r = torch.randn(M, N, device=DEV).bfloat16()
            y = linear(x, w, b, act=act, residual=r)
        torch.cuda.synchronize()
    finally:
        set_gemm_tile(0)
    ref = x.float() @ w.float().t()
    if act == 3:
        g = ref.view(M, N // 16, 2, 8)
        ref = (torch.nn.functional.silu(g[:, :, 0]) * g[:, :, 1]).reshape(M, N // 2)
    else:
        ref = ref + b
        ref = torch.relu(ref) if act == 1 else torch.nn.functional.gelu(ref) if act == 2 else ref
        ref = ref + r.float()
    assert _rel(y, ref) < 1e-2


@pytest.mark.parametrize("M,N,K", [(4400, 4208, 192), (4352, 4352, 768), (8192, 768, 768)])
@pytest.mark.parametrize("epi", ["res", "gelu", "silu_mul", "norm"])
@pytest.mark.parametrize("tile", [256, 255])
def test_gemm_bf16_256_many_tiles(M, N, K, epi, tile):
    """More 256^2 tiles than CUs (several waves of workgroups, edge tiles, odd
    K-tile counts) with every prefill epilogue, incl. the folded pre-norm, vs fp32."""
    from distributed_neural_networks_amd.ops.gemm import linear, set_gemm_tile
    torch.manual_seed(3)
    x = torch.randn(M, K, device=DEV).bfloat16()
    w = (torch.randn(N, K, device=DEV) * 0.05).bfloat16()
    b = torch.randn(N, device=DEV)
    r = torch.randn(M, N, device=DEV).bfloat16()
    rowstat = colsum = None
    if epi == "norm":  # folded pre-norm epilogue: v = rstd acc - mean rstd colsum
        mean, rstd = torch.randn(M, device=DEV), torch.rand(M, device=DEV) + 0.5
        rowstat = torch.stack([rstd, -mean * rstd], 1).contiguous()
        colsum = torch.randn(N, device=DEV)
    set_gemm_tile(tile)
    try:
        if epi == "silu_mul":
            y = linear(x, w, act="silu_mul")
        elif epi == "gelu":
            y = linear(x, w, b, act="gelu")
        elif epi == "res":
            y = linear(x, w, b, residual=r)
        else:
            y = linear(x, w, b, rowstat=rowstat, colsum=colsum)
        torch.cuda.synchronize()
    finally:
        set_gemm_tile(0)
    ref = x.float() @ w.float().t()
    if epi == "silu_mul":
        g = ref.view(M, N // 16, 2, 8)
        ref = (torch.nn.functional.silu(g[:, :, 0]) * g[:, :, 1]).reshape(M, N // 2)
    elif epi == "gelu":
        ref = torch.nn.functional.gelu(ref + b)
    elif epi == "res":
        ref = ref + b + r.float()
    else:
        ref = ref * rowstat[:, :1] + rowstat[:, 1:] * colsum + b
    assert _rel(y, ref) < 1e-2


@pytest.mark.parametrize("M,N,K", [(4400, 1536, 192), (300, 768, 768), (513, 2304, 3072)])
@pytest.mark.parametrize("dtype", ["bf16", "fp8mx"])
@pytest.mark.parametrize("tile", [256, 255])
def test_gemm_256_residual_tile_dma_bit_identical(M, N, K, dtype, tile):
    """The 256^2 / 256x128 residual epilogue with its residual tile moved by
    LDS-DMA (gemm_epilogue.h res_tile_dma, the default) writes exactly what the
    per-lane residual gathers wrote (anatomy bit 4), incl. partial M tiles."""
    from distributed_neural_networks_amd.ops._lib import lib, ptr, stream_ptr
    from distributed_neural_networks_amd.ops.gemm import linear, set_gemm_tile
    from distributed_neural_networks_amd.ops.fp8 import kpad_of, mx_scale_bytes, quant_rows_mx, quantize_weight
    torch.manual_seed(9)
    x = torch.randn(M, K, device=DEV).bfloat16()
    w = (torch.randn(N, K, device=DEV) * 0.05).bfloat16()
    b = torch.randn(N, device=DEV)
    r = torch.randn(M, N, device=DEV).bfloat16()
    L = lib()
    if dtype == "fp8mx":
        if M < 256 or tile != 256:
            pytest.skip("the MX path: 256^2 tiles, M >= 256")
        wq = quantize_weight(w.float(), torch.device(DEV))
        kp = kpad_of(K)
        qb = torch.empty(M, kp, dtype=torch.uint8, device=DEV)
        sx = torch.empty(mx_scale_bytes(M, kp), dtype=torch.uint8, device=DEV)
        quant_rows_mx(x, qb, sx)

        def run():
            o = torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
            assert L.gemm_fp8_mx(ptr(qb), ptr(sx), ptr(wq.q), ptr(wq.scale), ptr(o), N, ptr(b), ptr(r), N, M, N, kp,
                                 0, 0, 0, 0, 0, stream_ptr()) == 0
            return o
    else:
        def run():
            return linear(x, w, b, residual=r)
    set_gemm_tile(tile)
    try:
        outs = []
        for bits in (4, 0):
            assert L.gemm_set_anatomy(bits) == 0
            outs.append(run())
            torch.cuda.synchronize()
    finally:
        L.gemm_set_anatomy(0)
        set_gemm_tile(0)
    assert torch.equal(outs[0], outs[1])
    ref = x.float() @ w.float().t() + b + r.float()
    assert _rel(outs[1], ref) < (5e-2 if dtype == "fp8mx" else 1e-2)


@pytest.mark.parametrize("tile", [256, 255])
def test_gemm_256_asymmetric_layout(tile):
    from distributed_neural_networks_amd.ops.gemm import linear, set_gemm_tile
    n = 512
    x = torch.eye(n, device=DEV).bfloat16()
    w = torch.arange(n * n, device=DEV, dtype=torch.float32).reshape(n, n).remainder(97).bfloat16()
    set_gemm_tile(tile)
    try:
        y = linear(x, w, out_dtype=torch.float32)
        torch.cuda.synchronize()
    finally:
        set_gemm_tile(0)
    assert torch.equal(y, w.float().t())


def test_gemm_asymmetric_layout():
    """A = I with an asymmetric W catches a transposed C write (guide §3)."""
    from distributed_neural_networks_amd.ops.gemm import linear
    n = 128
    x = torch.eye(n, device=DEV).bfloat16()
    w = torch.arange(n * n, device=DEV, dtype=torch.float32).reshape(n, n).remainder(97).bfloat16()
    y = linear(x, w, out_dtype=torch.float32)
    assert torch.equal(y, w.float().t())


@pytest.mark.parametrize("tile", [128, 256])
@pytest.mark.parametrize("n", [512, 520])
def test_gemm_asymmetric_layout_bf16(tile, n):
    """bf16 output takes the widened (permlane16-swapped, 16-B) store path; an
    identity A with an asymmetric W pins every column of the swapped layout,
    and n = 520 leaves a 32-column group that falls back to 8-B stores."""
    from distributed_neural_networks_amd.ops.gemm import linear, set_gemm_tile
    k = 512
    x = torch.eye(k, device=DEV).bfloat16()
    w = torch.arange(n * k, device=DEV, dtype=torch.float32).reshape(n, k).remainder(97).bfloat16()
    set_gemm_tile(tile)
    try:
        y = linear(x, w)
        torch.cuda.synchronize()
    finally:
        set_gemm_tile(0)
    assert y.dtype == torch.bfloat16
    assert torch.equal(y, w.t())


def test_gemm_gelu_erf_accuracy():
    """The branch-free erf GELU epilogue vs torch's exact-erf GELU, element-wise
    (identity A, fp32 out): |error| must stay far below one bf16 ulp."""
    from distributed_neural_networks_amd.ops.gemm import linear
    n = 256
    x = torch.eye(n, device=DEV).bfloat16()
    w = torch.linspace(-12, 12, n * n, device=DEV).reshape(n, n).bfloat16()
    y = linear(x, w, act=2, out_dtype=torch.float32)
    ref = torch.nn.functional.gelu(w.float().t())
    assert (y - ref).abs().max().item() < 2e-6 * 12


@pytest.mark.parametrize("tile", [128, 256])
@pytest.mark.parametrize("M,N,K", [(300, 2048, 768), (1000, 528, 256), (4096, 1024, 512)])
def test_gemm_silu_mul_tiles(tile, M, N, K):
    """SwiGLU epilogue of the tiled GEMMs (paired-tile permlane32 exchange),
    forced 128^2 and 256^2, partial tiles included."""
    from distributed_neural_networks_amd.ops.gemm import linear, pack_gate_up, set_gemm_tile
    torch.manual_seed(5)
    x = torch.randn(M, K, device=DEV).bfloat16()
    g = (torch.randn(N // 2, K, device=DEV) * 0.05).bfloat16()
    u = (torch.randn(N // 2, K, device=DEV) * 0.05).bfloat16()
    set_gemm_tile(tile)
    try:
        y = linear(x, pack_gate_up(g, u), act="silu_mul")
        torch.cuda.synchronize()
    finally:
        set_gemm_tile(0)
    ref = torch.nn.functional.silu(x.float() @ g.float().t()) * (x.float() @ u.float().t())
    assert y.shape == (M, N // 2)
    assert _rel(y, ref) < 1e-2


def test_gemm_silu_mul():
    from distributed_neural_networks_amd.ops.gemm import linear, pack_gate_up
    torch.manual_seed(1)
    for M in (1, 5, 31, 64, 65, 200):
        x = torch.randn(M, 256, device=DEV).bfloat16()
        g = (torch.randn(512, 256, device=DEV) * 0.05).bfloat16()
        u = (torch.randn(512, 256, device=DEV) * 0.05).bfloat16()
        y = linear(x, pack_gate_up(g, u), act="silu_mul")
        ref = torch.nn.functional.silu(x.float() @ g.float().t()) * (x.float() @ u.float().t())
        assert y.shape == (M, 512)
        assert _rel(y, ref) < 1e-2


def _cifar_golden(seed, B):
    from distributed_neural_networks_amd.models.cifar import CifarStage, NeuralNetwork
    torch.manual_seed(seed)
    model = NeuralNetwork().eval()
    sd = model.state_dict()
    x = torch.randn(B, 3, 32, 32)
    with torch.no_grad():
        part0 = CifarStage(0, 1).eval()
        part0.load_state_dict(sd, strict=False)
        mid = part0(x)
        ref = model(x)
    return sd, x, mid, ref


@pytest.mark.parametrize("B", [1, 3, 64, 1000])
def test_cifar_stage0_and_head_bf16(B):
    from distributed_neural_networks_amd.ops import cifar as cops
    sd, x, mid, ref_out = _cifar_golden(0, B)
    w0 = cops.pack_stage0(sd, DEV, "bf16")
    wh = cops.pack_head(sd, DEV, precision="bf16")
    h = cops.stage0_forward(x.to(DEV), w0)
    torch.cuda.synchronize()
    assert h.dtype == torch.bfloat16
    assert _rel(h.cpu(), mid) < 1e-2
    probs, pred = cops.head_forward(h, wh)
    torch.cuda.synchronize()
    assert (probs.cpu() - ref_out).abs().max().item() < 2e-2
    assert (pred.cpu().long() == ref_out.argmax(1)).float().mean().item() > 0.9
    assert torch.equal(pred.cpu().long(), probs.cpu().argmax(1))


@pytest.mark.parametrize("B", [1, 3, 257, 1000])
def test_cifar_fp32_stage0_and_head(B):
    """fp32 path (3-term bf16 split on MFMA) against the fp32 torch stages."""
    from distributed_neural_networks_amd.ops import cifar as cops
    sd, x, mid, ref_out = _cifar_golden(1, B)
    w0 = cops.pack_stage0(sd, DEV)
    wh = cops.pack_head(sd, DEV)
    h = cops.stage0_forward(x.to(DEV), w0)
    torch.cuda.synchronize()
    assert h.dtype == torch.float32
    err = (h.cpu() - mid).abs().max().item()
    assert err <= 2e-5 * max(1.0, mid.abs().max().item()), err
    probs, pred = cops.head_forward(h, wh)
    torch.cuda.synchronize()
    assert (probs.cpu() - ref_out).abs().max().item() <= 1e-5
    assert torch.equal(pred.cpu().long(), probs.cpu().argmax(1))


@pytest.mark.parametrize("boundary", ["fp32", "split"])
def test_cifar_fp32_pipeline_4096_images_matches_reference(boundary):
    """Acceptance: the 2-stage pipeline at the reference's
    precision on 4096 images: max |dprob| <= 1e-5 vs fp32 torch
    (cifar_model_parts.py:7-26) and 100 % argmax agreement (rows whose golden
    top-2 probabilities tie within 1e-6 are excluded as numerically undecidable)."""
    from distributed_neural_networks_amd.runtime.pipeline import ColocatedPipeline
    from distributed_neural_networks_amd.runtime.stages import CifarHipStage
    sd, x, _, ref = _cifar_golden(2, 4096)
    st = [CifarHipStage(sd, 0, 1, DEV, boundary=boundary), CifarHipStage(sd, 2, 3, DEV, boundary=boundary)]
    assert st[0].out_spec(4) == ((4, 4096), torch.float32)
    out = ColocatedPipeline(st, 4096)(x.to(DEV))
    torch.cuda.synchronize()
    dp = (out.probs.cpu() - ref).abs().max().item()
    assert dp <= 1e-5, dp
    top2 = ref.topk(2, dim=1).values
    decidable = (top2[:, 0] - top2[:, 1]) > 1e-6
    agree = out.pred.cpu().long() == ref.argmax(1)
    assert bool(agree[decidable].all()), int((~agree[decidable]).sum())


@pytest.mark.parametrize("cut,precision", [(1, "fp32"), (2, "fp32"), (1, "bf16"), (2, "bf16")])
def test_cifar_stage_cuts(cut, precision):
    """Both 2-stage cuts (reference conv|fc and the fc1 cut) reproduce the full model."""
    from distributed_neural_networks_amd.models.cifar import NeuralNetwork
    from distributed_neural_networks_amd.runtime.pipeline import ColocatedPipeline
    from distributed_neural_networks_amd.runtime.stages import CifarHipStage
    torch.manual_seed(5)
    m = NeuralNetwork().eval()
    sd = m.state_dict()
    st = [CifarHipStage(sd, 0, cut, DEV, precision), CifarHipStage(sd, cut + 1, 3, DEV, precision)]
    x = torch.randn(64, 3, 32, 32)
    out = ColocatedPipeline(st, 64)(x.to(DEV))
    torch.cuda.synchronize()
    with torch.no_grad():
        ref = m(x)
    tol = 1e-5 if precision == "fp32" else 2e-2
    assert (out.probs.cpu() - ref).abs().max().item() < tol
    dt = torch.float32 if precision == "fp32" else torch.bfloat16
    assert st[0].out_spec(8) == ((8, 4096 if cut == 1 else 512), dt)


@pytest.mark.parametrize("split_in", [0, 1])
@pytest.mark.parametrize("M,N,K", [(300, 256, 64), (1000, 512, 4096), (16384 + 77, 512, 4096)])
def test_cifar_fc1_x3_kernel(M, N, K, split_in):
    """Fused fp32 fc1 (A split in registers while staging, or A in the blocked
    hi/lo encoding staged by DMA): relu(A W^T + b) vs fp32 torch, relative
    error at the ~2^-16 level of the 3-term split."""
    from distributed_neural_networks_amd.ops import _lib
    from distributed_neural_networks_amd.ops.cifar import encode_boundary, split_bf16
    torch.manual_seed(M)
    a = torch.randn(M, K, device=DEV)
    w = torch.randn(N, K, device=DEV) / K ** 0.5
    b = torch.randn(N, device=DEV) * 0.1
    wh, wl = split_bf16(w)
    out = torch.empty(M, N, device=DEV)
    a_in = encode_boundary(a) if split_in else a
    rc = _lib.lib().cifar_fc1_x3(a_in.data_ptr(), K, wh.data_ptr(), wl.data_ptr(), K, b.data_ptr(), out.data_ptr(),
                                 N, M, N, K, torch.cuda.current_stream().cuda_stream, split_in)
    assert rc == 0
    torch.cuda.synchronize()
    ref = torch.relu(a.double() @ w.double().t() + b.double())
    err = (out.double() - ref).abs().max().item()
    assert err <= 2e-5 * ref.abs().max().item(), err


@pytest.mark.parametrize("split_in", [0, 1])
@pytest.mark.parametrize("M,N,K,pad", [(1, 256, 32, 0), (255, 256, 64, 4), (257, 512, 96, 32), (600, 512, 160, 0)])
def test_cifar_fc1_x3_edges(M, N, K, pad, split_in):
    """One to five k-steps (the DMAs run up to two ahead and refill the last one past
    the end), rows past the matrix, rows of a wider tensor, the widest range of values
    a split takes.  Two terms of a product are off by 2^-16 of it, and K fp32 sums by
    K 2^-24: within 2^-14 of the sum of magnitudes."""
    from distributed_neural_networks_amd.ops import _lib
    from distributed_neural_networks_amd.ops.cifar import encode_boundary, split_bf16
    torch.manual_seed(M)
    a = torch.randn(M, K, device=DEV) * torch.exp2(torch.randint(-40, 40, (M, 1), device=DEV).float())
    w = torch.randn(N, K, device=DEV)
    b = torch.zeros(N, device=DEV)
    wh, wl = split_bf16(w)
    rows = torch.full((M, K + pad), float("nan"), device=DEV)
    rows[:, :K] = encode_boundary(a) if split_in else a
    out = torch.full((M + 1, N), 7.0, device=DEV)
    rc = _lib.lib().cifar_fc1_x3(rows.data_ptr(), K + pad, wh.data_ptr(), wl.data_ptr(), K, b.data_ptr(), out.data_ptr(),
                                 N, M, N, K, torch.cuda.current_stream().cuda_stream, split_in)
    assert rc == 0
    torch.cuda.synchronize()
    ref = torch.relu(a.double() @ w.double().t())
    bound = a.double().abs() @ w.double().abs().t() * 2 ** -14
    assert ((out[:M].double() - ref).abs() <= bound).all()
    assert (out[M] == 7).all()


@pytest.mark.parametrize("split_in", [0, 1])
@pytest.mark.parametrize("M,K,splits", [(1, 96, 3), (257, 160, 2), (600, 4096, 12), (1000, 416, 5)])
def test_cifar_fc1_x3_ranges(M, K, splits, split_in):
    """K in ranges of unequal and of one k-step, rows past the matrix; parts behind the
    ones asked for stay as they are.  Bound: test_cifar_fc1_x3_edges."""
    from distributed_neural_networks_amd.ops import _lib
    from distributed_neural_networks_amd.ops.cifar import encode_boundary, split_bf16
    torch.manual_seed(M)
    N = 256
    a, w, b = torch.randn(M, K, device=DEV), torch.randn(N, K, device=DEV), torch.randn(N, device=DEV)
    wh, wl = split_bf16(w)
    a_in = encode_boundary(a) if split_in else a
    out, part = torch.full((M + 1, N), 7.0, device=DEV), torch.full((splits * M * N + 64,), 7.0, device=DEV)
    rc = _lib.lib().cifar_fc1_x3(a_in.data_ptr(), K, wh.data_ptr(), wl.data_ptr(), K, b.data_ptr(), out.data_ptr(), N, M,
                                 N, K, torch.cuda.current_stream().cuda_stream, split_in, splits, part.data_ptr())
    assert rc == 0
    torch.cuda.synchronize()
    ref = torch.relu(a.double() @ w.double().t() + b.double())
    bound = (a.double().abs() @ w.double().abs().t() + b.double().abs()) * 2 ** -14
    assert ((out[:M].double() - ref).abs() <= bound).all()
    assert (out[M] == 7).all() and (part[splits * M * N:] == 7).all()


@pytest.mark.parametrize("B", [513, 1000, 8700, 9000, 16400])
def test_cifar_fc1_batches(B):
    """fc1 on every side of its rules, with the stage's scratch and its own, into plain, strided
    (16 bytes apart and not) and bf16 rows; what lies beside them stays.  bf16 has 8 significant
    bits: a result is rounded by at most 2^-8 of itself."""
    from distributed_neural_networks_amd.ops import cifar as cops
    torch.manual_seed(B)
    w = cops.pack_head({"fc1.weight": torch.randn(512, 4096) / 64, "fc1.bias": torch.randn(512), "fc2.weight": torch.randn(10, 512),
                        "fc2.bias": torch.randn(10)}, DEV)
    h = torch.rand(B, 4096, device=DEV)
    ref = torch.relu(h.double() @ (w.w_fc1h.double() + w.w_fc1l.double()).t() + w.b_fc1.double())
    rows = cops.fc1_scratch_rows(B)
    own = torch.empty((rows, 3 * 4096), dtype=torch.bfloat16, device=DEV) if rows else None
    outs = [cops.fc1_forward(h, w, scratch=own), cops.fc1_forward(h, w)]
    assert torch.equal(*outs)
    for cols in (520, 517):
        wide = torch.full((B + 1, cols), 7.0, device=DEV)
        outs.append(cops.fc1_forward(h, w, out=wide[:B, :512]))
        assert (wide[:, 512:] == 7).all() and (wide[B] == 7).all()
    typed = torch.full((B + 1, 512), 7.0, device=DEV, dtype=torch.bfloat16)
    y = cops.fc1_forward(h, w, out=typed[:B])
    assert ((y.double() - ref).abs() <= ref * 2 ** -8 + 2e-5 * ref.abs().max()).all() and (typed[B] == 7).all()
    for y in outs:
        assert (y.double() - ref).abs().max().item() <= 2e-5 * ref.abs().max().item()


@pytest.mark.parametrize("boundary", ["fp32", "split"])
@pytest.mark.parametrize("B", [513, 8704])
def test_cifar_fc1_rows_off_16_bytes(B, boundary):
    """Boundary rows that start one float behind a 16-byte address, against 64 bits
    (bound: test_cifar_fc1_x3_edges)."""
    from distributed_neural_networks_amd.ops import cifar as cops
    torch.manual_seed(B)
    w = cops.pack_head({"fc1.weight": torch.randn(512, 4096) / 64, "fc1.bias": torch.randn(512), "fc2.weight": torch.randn(10, 512),
                        "fc2.bias": torch.randn(10)}, DEV)
    a = torch.rand(B, 4096, device=DEV)
    h = torch.empty(B * 4096 + 1, device=DEV)[1:].view(B, 4096)
    h.copy_(cops.encode_boundary(a) if boundary == "split" else a)
    assert h.is_contiguous() and h.data_ptr() % 16 == 4
    y = cops.fc1_forward(h, w, boundary=boundary)
    W = w.w_fc1h.double() + w.w_fc1l.double()
    ref = torch.relu(a.double() @ W.t() + w.b_fc1.double())
    bound = (a.double() @ W.abs().t() + w.b_fc1.double().abs()) * 2 ** -14
    assert ((y.double() - ref).abs() <= bound).all()


@pytest.mark.parametrize("boundary", ["fp32", "split"])
@pytest.mark.parametrize("B", [1, 2, 15, 16, 17, 32, 33, 64, 65, 500, 512])
def test_cifar_few_images(B, boundary):
    """Bands of one image against whole images a workgroup (the same bits) and the
    head in slices of K against fp64: a product of the 3-term split is off by at
    most 2^-16 of itself, and 4096 + 512 fp32 sums stay below 2^-17 of the sum of
    magnitudes."""
    from distributed_neural_networks_amd.ops import cifar as cops
    assert B <= cops.FC1_FEW_ROWS
    sd, x, _, _ = _cifar_golden(B, B)
    w0, wh = cops.pack_stage0(sd, DEV), cops.pack_head(sd, DEV)
    x = x.to(DEV)
    h = cops.stage0_forward(x, w0, boundary=boundary)
    whole = cops.stage0_forward(x, w0, grid=B, boundary=boundary)  # B workgroups: no bands
    assert torch.equal(h, whole)
    hid = torch.full((B, 512), float("nan"), device=DEV)
    probs, pred = cops.head_forward(h, wh, hid=hid, boundary=boundary)
    alone = cops.fc1_forward(h, wh, boundary=boundary)
    assert torch.equal(hid, alone)
    p2, k2 = cops.head_forward(h, wh, boundary=boundary)
    assert torch.equal(probs, p2) and torch.equal(pred, k2)
    hv = cops.decode_boundary(h) if boundary == "split" else h
    W, b = sd["fc1.weight"].to(DEV).double(), sd["fc1.bias"].to(DEV).double()
    ref = torch.relu(hv.double() @ W.t() + b)
    bound = (hv.double().abs() @ W.abs().t() + b.abs()) * 3 * 2.0 ** -17
    assert bool(((hid.double() - ref).abs() <= bound).all())
    W2, b2 = sd["fc2.weight"].to(DEV).double(), sd["fc2.bias"].to(DEV).double()
    z = hid.double() @ W2.t() + b2
    err = (hid.double() @ W2.abs().t() + b2.abs()).max() * 2.0 ** -16
    assert (probs.double() - z.softmax(1)).abs().max() <= err + 2.0 ** -20
    assert torch.equal(pred.long(), probs.argmax(1))


def _stage0_in_64_bits(sd, x):
    """(units 0-1, the sums of magnitudes behind them, conv1's share of those) in float64."""
    def conv(t, w, b):
        n, _, h, _ = t.shape
        u = torch.nn.functional.pad(t, (1, 1, 1, 1)).unfold(2, 3, 1).unfold(3, 3, 1)
        y = u.permute(0, 2, 3, 1, 4, 5).reshape(n * h * h, -1) @ w.reshape(w.shape[0], -1).t() + b
        return y.view(n, h, h, -1).permute(0, 3, 1, 2)
    W = {k: v.to(DEV).double() for k, v in sd.items()}
    x = x.to(DEV).double()
    pool = torch.nn.functional.max_pool2d
    a = pool(conv(x, W["conv1.weight"], W["conv1.bias"]).relu(), 2)
    mag = pool(conv(x.abs(), W["conv1.weight"].abs(), W["conv1.bias"].abs()), 2)
    y = pool(conv(a, W["conv2.weight"], W["conv2.bias"]).relu(), 2)
    own = conv(mag, W["conv2.weight"].abs(), W["conv2.bias"].abs())
    # the 4 x 4 patch of every output: F(2 x 2, 3 x 3) meets all of it
    patch = torch.nn.functional.max_pool2d(torch.nn.functional.pad(mag, (1, 1, 1, 1)), 4, 2)
    wide = patch.permute(0, 2, 3, 1) @ W["conv2.weight"].abs().sum((2, 3)).t()
    return y.flatten(1), pool(own, 2).flatten(1), wide.permute(0, 3, 1, 2).flatten(1)


@pytest.mark.parametrize("boundary", ["fp32", "split"])
@pytest.mark.parametrize("B,grid,kind", [(3, 1, "plain"), (5, 2, "plain"), (7, 2, "holes"), (7, 3, "wide"), (513, 0, "plain"),
                                         (1025, 256, "holes"), (4, 1, "huge"), (6, 2, "flat")])
def test_cifar_winograd(B, grid, kind, boundary):
    """conv2 by Winograd against 64 bits and against the direct form: workgroups with 3 and more images, and
    with unequal numbers of them; infinities and NaN (what they reach is 0 in both forms); a range too wide for
    one scale (the direct form's bits); images of magnitudes near the range's ends.  Bound: conv1 is off by 3 * 2^-17
    of its magnitudes; a product of conv2 by 2^-19, of which an output sums 9 of operands up to 4 times the patch's."""
    from distributed_neural_networks_amd.ops import cifar as cops
    g = torch.Generator().manual_seed(B)
    sd, _, _, _ = _cifar_golden(B, 1)
    x = torch.randn(B, 3, 32, 32, generator=g) * {"huge": 500.0, "flat": 1e-6}.get(kind, 1.0)
    if kind == "holes":
        x[0, 1, 0, 0], x[1, 0, 31, 31], x[2, 2, 13, 18], x[-1, 1, 16, 7] = float("inf"), float("nan"), -float("inf"), float("nan")
    if kind == "wide":
        x[::2, :, :16] *= 1e6
    w0, x = cops.pack_stage0(sd, DEV), x.to(DEV)
    assert w0.u2h is not None and B > cops.WINO_ROUNDS * (grid or 256)
    keep, h = torch.zeros_like(x), torch.full((B, 4096), float("nan"), device=DEV)
    cops.stage0_forward(x, w0, h, grid=grid, boundary=boundary, keep=keep)
    assert torch.equal(keep.view(torch.int32), x.view(torch.int32))
    direct = cops.stage0_forward(x, w0, grid=B, boundary=boundary)  # one image a workgroup
    if boundary == "split":
        plain = cops.stage0_forward(x, w0, grid=grid)
        assert torch.equal(cops.encode_boundary(plain).view(torch.int32), h.view(torch.int32))
        h, direct = plain, cops.decode_boundary(direct)
    if kind == "wide":
        assert torch.equal(h[::2], cops.stage0_forward(x, w0, grid=B)[::2])
    if kind == "holes":
        clean = torch.nan_to_num(x, nan=0.0, posinf=0.0, neginf=0.0)
        touched = torch.nn.functional.pad((x != clean).any(1, keepdim=True).float(), (1, 2, 1, 1))
        touched = torch.nn.functional.max_pool2d(touched, (3, 4), 1)  # conv1's windows, whose rows are padded to 4 with zeros
        touched = torch.nn.functional.max_pool2d(touched, 2)
        touched = torch.nn.functional.max_pool2d(torch.nn.functional.max_pool2d(touched, 3, 1, 1), 2)
        away = (touched == 0).expand(B, 64, 8, 8).reshape(B, 4096)
        ref, own, wide = _stage0_in_64_bits(sd, clean)
        assert ((h - direct).abs() <= own * 3 * 2.0 ** -16 + wide * 36 * 2.0 ** -18).all()  # 0 for 0 where they reach
        ref, own, wide = (t * away for t in (ref, own, wide))
        h, direct = h * away, direct * away
    else:
        ref, own, wide = _stage0_in_64_bits(sd, x)
    assert ((h.double() - ref).abs() <= own * 3 * 2.0 ** -17 + wide * 36 * 2.0 ** -19).all()
    assert (h.double() - ref).norm() <= 1.05 * (direct.double() - ref).norm()  # no further off than the direct form


def test_cifar_without_biases_stays_direct():
    """Without biases beside them, small parts of an image have no floor: the direct form, the same bits."""
    from distributed_neural_networks_amd.ops import cifar as cops
    sd, x, _, _ = _cifar_golden(5, 5)
    sd = {k: torch.zeros_like(v) if k == "conv1.bias" else v for k, v in sd.items()}
    w0, x = cops.pack_stage0(sd, DEV), x.to(DEV)
    assert w0.u2h is None
    assert torch.equal(cops.stage0_forward(x, w0, grid=1), cops.stage0_forward(x, w0, grid=5))


def _spread(kind, sd):
    sd = {k: v.clone() for k, v in sd.items()}
    if kind in ("bias", "dead"):  # one channel's bias, which half of the outputs do not read
        sd["conv1.bias"][3] = 1e7 if kind == "bias" else -1e7
        sd["conv2.weight"][::2, 3] = 0
    if kind == "weights":  # one channel small in conv1 and large in conv2
        for k in ("conv1.weight", "conv1.bias"):
            sd[k][3] *= 2.0 ** -24
        sd["conv2.weight"][:, 3] *= 2.0 ** 24
    if kind == "little":  # images beyond 40 reach past the range beside these biases
        sd["conv1.bias"] *= 0.02
    if kind == "none":
        sd["conv2.weight"].zero_()
    if kind == "holes":  # a filter of zeros loses nothing, a lost channel bounds nothing
        sd["conv2.weight"][5, 7] = 0
        sd["conv1.weight"][9, 0, 1, 1], sd["conv1.bias"][11] = float("inf"), float("nan")
    return sd


@pytest.mark.parametrize("kind,takes", [("plain", True), ("none", True), ("holes", True), ("bias", False), ("dead", False),
                                        ("weights", False), ("little", False)])
def test_cifar_winograd_takes_weights(kind, takes):
    """Weights of a spread that one scale an image or an output channel would cut bits of stay with the direct form; where
    they do not, conv2 of few images and of many is as close to 64 bits (bounds: test_cifar_winograd)."""
    from distributed_neural_networks_amd.ops import cifar as cops
    sd, x, _, _ = _cifar_golden(5, 5)
    sd = _spread(kind, sd)
    w0, x = cops.pack_stage0(sd, DEV), x.to(DEV)
    h = cops.stage0_forward(x, w0, grid=1)
    if kind != "holes":
        ref, own, wide = _stage0_in_64_bits(sd, x)
        assert ((h.double() - ref).abs() <= own * 3 * 2.0 ** -17 + wide * 36 * 2.0 ** -19).all()
    assert (w0.u2h is not None) == takes


def test_cifar_winograd_raw_pixels():
    """Images of 0 to 255 are in range: Winograd's form (other bits than the direct one), the bounds of test_cifar_winograd."""
    from distributed_neural_networks_amd.ops import cifar as cops
    sd, x, _, _ = _cifar_golden(6, 6)
    x = torch.randint(0, 256, x.shape, generator=torch.Generator().manual_seed(6)).float()
    x[:, :, 8:20, 8:20] = 0
    w0, x = cops.pack_stage0(sd, DEV), x.to(DEV)
    h, direct = (cops.stage0_forward(x, w0, grid=g) for g in (2, 6))
    ref, own, wide = _stage0_in_64_bits(sd, x)
    assert ((h.double() - ref).abs() <= own * 3 * 2.0 ** -17 + wide * 36 * 2.0 ** -19).all()
    assert all(not torch.equal(a, b) for a, b in zip(h, direct))
    assert (h.double() - ref).norm() <= 1.05 * (direct.double() - ref).norm()


@pytest.mark.parametrize("boundary", ["fp32", "split"])
def test_cifar_fp32_pipeline_large_batch_fused_fc1(boundary):
    """The large-batch fp32 head (fused fc1) on 20000 images: max |dprob| <= 1e-5
    vs the fp32 torch model and argmax agreement on every decidable row."""
    from distributed_neural_networks_amd.ops import cifar as cops
    from distributed_neural_networks_amd.runtime.pipeline import ColocatedPipeline
    from distributed_neural_networks_amd.runtime.stages import CifarHipStage
    B = 20000
    assert B >= cops.FC1_X3_MIN_ROWS
    sd, x, _, ref = _cifar_golden(3, B)
    st = [CifarHipStage(sd, 0, 1, DEV, boundary=boundary), CifarHipStage(sd, 2, 3, DEV, boundary=boundary)]
    out = ColocatedPipeline(st, B)(x.to(DEV))
    torch.cuda.synchronize()
    dp = (out.probs.cpu() - ref).abs().max().item()
    assert dp <= 1e-5, dp
    top2 = ref.topk(2, dim=1).values
    decidable = (top2[:, 0] - top2[:, 1]) > 1e-6
    agree = out.pred.cpu().long() == ref.argmax(1)
    assert bool(agree[decidable].all()), int((~agree[decidable]).sum())


@pytest.mark.parametrize("B", [1, 300, 16384 + 77])
def test_cifar_split_boundary_bit_identical(B):
    """The blocked hi/lo boundary encoding is exactly the split of the fp32
    boundary (stage-0 epilogue == encode of the fp32 output, bitwise), decodes
    to it within 2^-16, and the pipeline's probabilities and predictions are
    bitwise those of the fp32 boundary (small-batch split3 path and the fused
    fc1 path)."""
    from distributed_neural_networks_amd.ops import cifar as cops
    from distributed_neural_networks_amd.runtime.pipeline import ColocatedPipeline
    from distributed_neural_networks_amd.runtime.stages import CifarHipStage
    torch.manual_seed(B)
    from distributed_neural_networks_amd.models.cifar import NeuralNetwork
    sd = NeuralNetwork().state_dict()
    x = torch.randn(B, 3, 32, 32, device=DEV)
    w0 = cops.pack_stage0(sd, DEV, "fp32")
    h32 = cops.stage0_forward(x, w0, boundary="fp32")
    hsp = cops.stage0_forward(x, w0, boundary="split")
    assert torch.equal(cops.encode_boundary(h32).view(torch.int32), hsp.view(torch.int32))
    back = cops.decode_boundary(hsp)
    assert ((back - h32).abs() <= h32.abs() * 2 ** -16).all()
    outs = {}
    for bd in ("fp32", "split"):
        st = [CifarHipStage(sd, 0, 1, DEV, boundary=bd), CifarHipStage(sd, 2, 3, DEV, boundary=bd)]
        o = ColocatedPipeline(st, B)(x)
        outs[bd] = (o.probs.clone(), o.pred.clone())
    torch.cuda.synchronize()
    assert torch.equal(outs["fp32"][0], outs["split"][0])
    assert torch.equal(outs["fp32"][1], outs["split"][1])


@pytest.mark.parametrize("K,act,res,fold", [(768, None, True, False), (3072, None, True, False),
                                            (768, "gelu", False, False), (768, None, False, True)])
def test_gemm_tail_split_matches_single_grid(K, act, res, fold):
    """GPT-2's 768-wide prefill projections at M = 32768 run as 256^2 tiles on
    the first 512 columns plus 256x128 tiles on the last 256 (two launches,
    disjoint columns): identical to the single 256^2 grid (same per-output
    MFMA order), with bias, residual, activation and the folded-norm epilogue,
    and close to fp32."""
    from distributed_neural_networks_amd.ops import transformer_ops as T
    from distributed_neural_networks_amd.ops.gemm import linear, set_gemm_split_tail, set_gemm_tile
    M, N = 32768, 768
    g = torch.Generator(device=DEV).manual_seed(4)
    x = torch.randn(M, K, device=DEV, generator=g).bfloat16()
    w = (torch.randn(N, K, device=DEV, generator=g) / K ** 0.5).bfloat16()
    b = torch.randn(N, device=DEV, generator=g) * 0.1
    r = torch.randn(M, N, device=DEV, generator=g).bfloat16() if res else None
    kw = {}
    if fold:
        st = torch.empty((M, 2), device=DEV, dtype=torch.float32)
        T.row_stats(x, st, 1e-5, False, rows=M, ldx=K)
        kw = dict(rowstat=st, colsum=w.float().sum(1).contiguous())
    outs = []
    try:
        for tile, split in ((0, True), (256, False)):
            set_gemm_tile(tile)
            set_gemm_split_tail(split)
            outs.append(linear(x, w, b, act, r, **kw))
            torch.cuda.synchronize()
    finally:
        set_gemm_tile(0)
        set_gemm_split_tail(True)
    assert torch.equal(outs[0], outs[1])
    xf = x.float()
    if fold:
        xf = torch.nn.functional.layer_norm(xf, (K,), eps=1e-5)
    ref = xf @ w.float().t() + b
    if act == "gelu":
        ref = torch.nn.functional.gelu(ref)
    if res:
        ref = ref + r.float()
    err = ((outs[0].float() - ref).norm() / ref.norm()).item()
    assert err < 1e-2, err


@pytest.mark.parametrize("N,K,split,act,res", [(1600, 1600, True, 0, True), (6400, 1600, True, 2, False),
                                               (1600, 6400, False, 0, True), (4800, 1600, True, 0, False)])
def test_fp8_gemm_tail_split_matches_single_grid(N, K, split, act, res):
    """GPT-2 XL prefill shapes on the fp8 256^2 kernel at M = 32768: the grid's
    last column of tiles (64 / 256 / 192 wide) as 256x128 tiles in a second
    launch gives the single grid's bits (split activations or not, GELU,
    residual)."""
    from distributed_neural_networks_amd.ops.fp8 import attach_split, linear_fp8, quantize_weight
    from distributed_neural_networks_amd.ops.gemm import set_gemm_split_tail
    M = 32768
    g = torch.Generator(device=DEV).manual_seed(6)
    x = torch.randn(M, K, device=DEV, generator=g).bfloat16()
    w = quantize_weight(torch.randn(N, K, device=DEV, generator=g) / K ** 0.5, DEV)
    if split:
        attach_split(w)
    b = torch.randn(N, device=DEV, generator=g) * 0.1
    r = torch.randn(M, N, device=DEV, generator=g).bfloat16() if res else None
    outs = []
    try:
        for mask in (3, 0):  # fp8 split on (off by default) / off
            set_gemm_split_tail(mask)
            outs.append(linear_fp8(x, w, b, act, r))
            torch.cuda.synchronize()
    finally:
        set_gemm_split_tail(True)
    assert torch.equal(outs[0], outs[1])
    ref = x.float() @ (w.q[:, :K].float() * w.scale[:, None]).t() + b
    if act == 2:
        ref = torch.nn.functional.gelu(ref)
    if res:
        ref = ref + r.float()
    err = ((outs[0].float() - ref).norm() / ref.norm()).item()
    assert err < (3e-2 if split else 8e-2), err


MID_TILES = ((64, 64), (128, 64), (128, 128), (256, 128), (128, 256), (192, 128), (96, 128))  # csrc/kernels/gemm_mid.hip MID


def _mid_reference(x, w, b, r, act, norm, consts):
    y = x.float() @ w.float().t()
    if norm is not None:
        st, cs = norm
        y = y * st[:, :1] + st[:, 1:] * cs
    if act in (3, 4):  # packed gate | up
        g = y.view(y.shape[0], -1, 2, 8)
        f = torch.nn.functional.silu if act == 3 else lambda z: torch.nn.functional.gelu(z, approximate="tanh")
        return (f(g[:, :, 0]) * g[:, :, 1]).reshape(y.shape[0], -1)
    if b is not None:
        y = y + b
    if act == 1:
        y = torch.relu(y)
    elif act == 2:
        y = torch.nn.functional.gelu(y)
    elif act == 6:
        y = torch.where(y > 0, consts[0] * y * y, consts[1] * (torch.expm1(y.clamp(max=0)) - y)) + y / 2
    return y if r is None else y + r.float()


@pytest.mark.parametrize("tile", range(5))
@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("dm,dn,K", [(1, 36, 192), (0, 0, 448), (-1, -8, 576), (3, 20, 4096)])
def test_gemm_mid_tiles(tile, splits, dm, dn, K):
    """Every tile of the mid-size GEMM, whole and with K over three workgroups, at
    sizes around its borders: plain, bias, activations, residual, gated, folded
    norm and fp32 outputs, strided operands and rows that no vector store fits.
    Inputs are bf16 and sums fp32, so a result is off by its rounding to bf16 (2^-9
    at most, 1.1e-3 rms) and an fp32 one by the order of its sums."""
    from distributed_neural_networks_amd.ops import gemm as G
    bm, bn = MID_TILES[tile]
    M, N = bm * (2 if bm == 64 else 1) + dm, bn + dn
    g = torch.Generator(device=DEV).manual_seed(tile * 10 + splits)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)  # noqa: E731
    x, w = rnd(M, K + 8).bfloat16()[:, :K], (rnd(N, K + 16) * K ** -0.5).bfloat16()[:, :K]
    b, ws = rnd(N), torch.zeros((4 * 3 * M * 2 * N) + 4096, dtype=torch.uint8, device=DEV)
    st, cs = torch.rand(M, 2, device=DEV, generator=g) + 0.5, w.float().sum(1).contiguous()
    r, odd = rnd(M, N).bfloat16(), torch.empty((M, N + 3), dtype=torch.bfloat16, device=DEV)[:, :N]
    consts = torch.tensor([0.7, 1.3], device=DEV)
    wg = (rnd(2 * (-(-N // 16) * 16), K) * K ** -0.5).bfloat16()
    calls = [(dict(bias=b, act=a, residual=r), w, b, r, a, None) for a in (0, 1, 2)]
    calls += [(dict(rowstat=st, colsum=cs, bias=b), w, b, None, 0, (st, cs)), (dict(out_dtype=torch.float32), w, None, None, 0, None),
              (dict(bias=torch.cat([b, consts]), act=6), w, b, None, 6, None), (dict(out=odd, residual=r), w, None, r, 0, None),
              (dict(act=3), wg, None, None, 3, None), (dict(act=4), wg, None, None, 4, None)]
    G.set_gemm_mid(tile, splits)
    try:
        for kw, wt, bias, res, act, norm in calls:
            y = G.linear(x, wt, ws=ws, **kw)
            assert torch.isfinite(y).all()
            assert _rel(y, _mid_reference(x, wt, bias, res, act, norm, consts)) < (1e-5 if y.dtype == torch.float32 else 2.5e-3), kw.keys()
    finally:
        G.set_gemm_mid()
    assert not ws[-4096:].any()  # the tickets of a decode workspace are not parts


@pytest.mark.parametrize("tile", [5, 6])
@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("dm,dn,K", [(1, 36, 192), (0, 0, 448), (-1, -8, 576), (-97, 20, 4096), (-47, 100, 320)])
def test_gemm_mid_tiles_between(tile, splits, dm, dn, K):
    """The tiles of 192 and 96 rows: as test_gemm_mid_tiles, and with rows that end in any wave's part."""
    test_gemm_mid_tiles(tile, splits, max(dm, 1 - MID_TILES[tile][0]), dn, K)


@pytest.mark.parametrize("M,N,K", [(65, 768, 3072), (96, 4096, 14336), (200, 6144, 4096), (256, 768, 768), (257, 4800, 1600),
                                   (700, 4096, 14336), (1071, 2304, 768), (4097, 768, 3072)])
@pytest.mark.parametrize("room", [0, 1 << 22, 1 << 26])
def test_gemm_chosen_tiles(M, N, K, room):
    """The tile, split or decode kernel that the estimate picks, with and without room for parts."""
    from distributed_neural_networks_amd.ops import gemm as G
    g = torch.Generator(device=DEV).manual_seed(M)
    x, w = torch.randn(M, K, device=DEV, generator=g).bfloat16(), torch.randn(N, K, device=DEV, generator=g).bfloat16()
    w = (w.float() * K ** -0.5).bfloat16()
    ws = torch.zeros(room + 4096, dtype=torch.uint8, device=DEV) if room else None
    for sh in (None, G.shuffle_weight(w)):
        assert _rel(G.linear(x, w, ws=ws, w_shuf=sh), x.float() @ w.float().t()) < 2.5e-3


@pytest.mark.parametrize("M", [9, 16, 17])
@pytest.mark.parametrize("N,K", [(20, 64), (4096, 192), (4112, 2048), (16384, 1984), (16400, 2048)])
def test_gemm_9_to_16_rows(M, N, K):
    """Either side of the lines of the 9 to 16 row rule: bf16 row-major and in fragment order, e4m3 weights.
    Tolerances: test_gemm_mid_tiles (the e4m3 product is exact in its weights)."""
    from distributed_neural_networks_amd.ops import gemm as G
    from distributed_neural_networks_amd.ops.fp8 import linear_w8, quantize_weight
    g = torch.Generator(device=DEV).manual_seed(M + N)
    x, w = torch.randn(M, K, device=DEV, generator=g).bfloat16(), torch.randn(N, K, device=DEV, generator=g) * K ** -0.5
    b, r = torch.randn(N, device=DEV, generator=g), torch.randn(M, N, device=DEV, generator=g).bfloat16()
    wb = w.bfloat16()
    ref = x.float() @ wb.float().t() + b + r.float()
    for sh in (None, G.shuffle_weight(wb)):
        assert _rel(G.linear(x, wb, b, residual=r, w_shuf=sh), ref) < 2.5e-3
    w8 = quantize_weight(w, DEV)
    ref8 = x.float() @ (w8.q[:, :K].float() * w8.scale[:, None]).t() + b + r.float()
    for _ in range(2):
        assert _rel(linear_w8(x, w8, b, residual=r), ref8) < 2.5e-3
        G.attach_shuffled(w8)


@pytest.mark.parametrize("M", [80, 81, 113, 129, 193, 208, 209, 240, 241, 256])
@pytest.mark.parametrize("N,K", [(1040, 64), (4092, 192), (4112, 448), (1600, 1600), (4092, 1600), (4112, 1600)])
def test_gemm_w8_65_to_256_rows(M, N, K):
    """16 rows a workgroup (the first three sizes) and either side of the rule to 64 rows, on 2 and on 4 column
    tiles (K of 1600), a last group of one row, columns cut inside a tile: e4m3 weights with bias and residual, GELU behind a folded norm, row-major
    and in fragment order.  Tolerances: test_gemm_9_to_16_rows."""
    from distributed_neural_networks_amd.ops import gemm as G
    from distributed_neural_networks_amd.ops.fp8 import linear_w8, quantize_weight
    g = torch.Generator(device=DEV).manual_seed(M + N)
    x, w = torch.randn(M, K, device=DEV, generator=g).bfloat16(), torch.randn(N, K, device=DEV, generator=g) * K ** -0.5
    b, r = torch.randn(N, device=DEV, generator=g), torch.randn(M, N, device=DEV, generator=g).bfloat16()
    w8 = quantize_weight(w, DEV)
    wd = w8.q[:, :K].float() * w8.scale[:, None]
    xn = torch.nn.functional.layer_norm(x.float(), (K,), eps=1e-5)
    ref, gelu = x.float() @ wd.t() + b + r.float(), torch.nn.functional.gelu(xn @ wd.t() + b)
    for _ in range(2):
        assert _rel(linear_w8(x, w8, b, residual=r), ref) < 2.5e-3
        assert _rel(linear_w8(x, w8, b, act=2, norm=2, colsum=wd.sum(1), eps=1e-5), gelu) < 2.5e-3
        G.attach_shuffled(w8)


@pytest.mark.parametrize("M,N,K", [(700, 22064, 768), (700, 22068, 2048), (1600, 12352, 2048)])
def test_gemm_columns_in_two(M, N, K):
    """Sizes whose columns are full rounds of 256 x 256 tiles and a rest on smaller ones (whole or
    split over K): every operand of the rest starts at its column.  Tolerances: test_gemm_mid_tiles."""
    from distributed_neural_networks_amd.ops import gemm as G
    g = torch.Generator(device=DEV).manual_seed(M)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)  # noqa: E731
    x, w, b, r = rnd(M, K).bfloat16(), (rnd(N, K) * K ** -0.5).bfloat16(), rnd(N), rnd(M, N).bfloat16()
    ws = torch.zeros((64 << 20) + 4096, dtype=torch.uint8, device=DEV)
    st, cs = torch.rand(M, 2, device=DEV, generator=g) + 0.5, w.float().sum(1).contiguous()
    consts = torch.tensor([0.7, 1.3], device=DEV)
    calls = [(dict(bias=b, act=2, residual=r), b, r, 2, None), (dict(rowstat=st, colsum=cs, bias=b), b, None, 0, (st, cs)),
             (dict(out_dtype=torch.float32, bias=b), b, None, 0, None), (dict(bias=torch.cat([b, consts]), act=6), b, None, 6, None)]
    if N % 16 == 0:
        calls += [(dict(act=3), None, None, 3, None), (dict(act=4), None, None, 4, None)]
    for kw, bias, res, act, norm in calls:
        y = G.linear(x, w, ws=ws, **kw)
        ref = _mid_reference(x, w, bias, res, act, norm, consts)
        tol = 1e-5 if y.dtype == torch.float32 else 2.5e-3
        for cols in (slice(0, 64), slice(y.shape[1] - 64, None), slice(None)):
            assert _rel(y[:, cols], ref[:, cols]) < tol, kw.keys()


@pytest.mark.parametrize("M,N,K", [(65, 2304, 768), (200, 4096, 4096), (256, 768, 3072), (128, 24448, 64), (200, 6144, 160),
                                   (256, 4096, 1056), (256, 2048, 8224), (256, 2048, 8256), (65, 24576, 64)])
@pytest.mark.parametrize("buffers", [False, True])
def test_linear_norm_65_to_256_rows(M, N, K, buffers):
    """Up to 191 tiles of 128 x 128 a folded norm runs on the decode kernels where the tiles cannot take it: without
    buffers, K of whole 32s, rows wider than the statistics kernel's; and a scatter says that it does not apply.
    Tolerance: bf16 products with fp32 sums and the result's rounding, the norm off by its rounding in fp32."""
    from distributed_neural_networks_amd.ops import gemm as G
    g = torch.Generator(device=DEV).manual_seed(M + K)
    x = torch.randn(M, K, device=DEV, generator=g).bfloat16()
    f = G.fold_norm(torch.randn(N, K, device=DEV, generator=g) * K ** -0.5, torch.ones(K, device=DEV), torch.zeros(K, device=DEV),
                    torch.randn(N, device=DEV, generator=g), False, 1e-5, DEV)
    kw = dict(std_buf=torch.empty(M, K, device=DEV, dtype=torch.bfloat16), ones=torch.ones(K, device=DEV)) if buffers else {}
    ref = torch.nn.functional.layer_norm(x.float(), (K,), eps=1e-5) @ f.w.float().t() + f.bias
    for ws in (None, G.shuffle_weight(f.w)):
        f.ws = ws
        if not buffers and -(-M // 128) * -(-N // 128) >= 192:
            continue
        assert _rel(G.linear_norm(x, f, **kw), ref) < 4e-3
        if buffers and -(-M // 128) * -(-N // 128) >= 192:  # an activation that only the tiles have
            assert _rel(G.linear_norm(x, f, act="relu", **kw), torch.relu(ref)) < 4e-3
    if buffers and (K % 64 or K > 8192):
        q, cache = torch.empty(M * N, device=DEV, dtype=torch.bfloat16), torch.empty(1, 1, M, 16, device=DEV, dtype=torch.bfloat16)
        H = N // 16 - 2
        assert not G.qkv_scatter_norm(x, f, kw["std_buf"], q, cache, cache.clone(), torch.zeros(1, device=DEV, dtype=torch.int32), 1, M,
                                      H, 1, 16)


@pytest.mark.parametrize("M,N,K", [(65, 2304, 768), (200, 4096, 1024), (256, 768, 3072), (130, 12544, 64)])
def test_gemm_65_to_256_rows_off_16_bytes(M, N, K):
    """Operands that start off 16 bytes or whose rows do: plain loads (the decode kernels) instead of the
    tiles' LDS-DMA.  Tolerance: test_gemm_mid_tiles."""
    from distributed_neural_networks_amd.ops import gemm as G
    g = torch.Generator(device=DEV).manual_seed(M + K)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g).bfloat16()  # noqa: E731
    x0, w0 = rnd(M * K + 3), rnd(N * K + 1)
    xs = [x0[3:].view(M, K), rnd(M, K + 5)[:, :K], rnd(M, K + 8)[:, 1:K + 1], rnd(M, K)]
    ws = [rnd(N, K)] * 3 + [w0[1:].view(N, K)]
    few = -(-M // 128) * -(-N // 128) < 192
    f = G.fold_norm(ws[0].float(), torch.ones(K, device=DEV), torch.zeros(K, device=DEV), None, False, 1e-5, DEV)
    for x, w in zip(xs, ws):
        w = (w.float() * K ** -0.5).bfloat16() if w.data_ptr() % 16 == 0 else w
        assert _rel(G.linear(x, w), x.float() @ w.float().t()) < 2.5e-3
        if few:
            ref = torch.nn.functional.layer_norm(x.float(), (K,), eps=1e-5) @ f.w.float().t()
            y = G.linear_norm(x, f, std_buf=torch.empty(M, K, device=DEV, dtype=torch.bfloat16), ones=torch.ones(K, device=DEV))
            assert _rel(y, ref) < 4e-3


@pytest.mark.parametrize("B,T,H,Hkv,hd,pos0,S", [(1, 65, 12, 12, 64, 0, 80), (3, 43, 4, 2, 128, 5, 60), (1, 255, 25, 25, 64, 9, 300)])
def test_qkv_scatter_small_prefill(B, T, H, Hkv, hd, pos0, S):
    """Fewer rows than a 256 x 256 tile: scattered on every small tile == qkv rows + qkv_split."""
    from distributed_neural_networks_amd.ops import gemm as G
    from distributed_neural_networks_amd.ops import transformer_ops as T_
    g = torch.Generator(device=DEV).manual_seed(B * T)
    d, N = 320, (H + 2 * Hkv) * hd
    x = torch.randn(B * T, d, device=DEV, generator=g).bfloat16()
    f = G.fold_norm(torch.randn(N, d, device=DEV, generator=g) * 0.05, torch.ones(d, device=DEV), torch.zeros(d, device=DEV),
                    torch.randn(N, device=DEV, generator=g) * 0.02, False, 1e-5, DEV)
    std, pos = torch.empty(B * T, d, device=DEV, dtype=torch.bfloat16), torch.full((B,), pos0, device=DEV, dtype=torch.int32)
    for tile in range(5):
        caches = [torch.zeros(B, Hkv, S, hd, device=DEV).bfloat16() for _ in range(4)]
        q, q2 = (torch.empty(B * H * T * hd, device=DEV, dtype=torch.bfloat16) for _ in range(2))
        G.set_gemm_mid(tile)
        try:
            assert G.qkv_scatter_norm(x, f, std, q, caches[0], caches[1], pos, B, T, H, Hkv, hd)
            qkv = G.linear_norm(x, f, std_buf=std, ones=torch.ones(d, device=DEV))
        finally:
            G.set_gemm_mid()
        T_.qkv_split(qkv, q2, caches[2], caches[3], B, T, H, Hkv, hd, pos)
        keep = pos0 + torch.arange(T, device=DEV) < S
        assert torch.equal(q.view(B, H, T, hd)[:, :, keep], q2.view(B, H, T, hd)[:, :, keep])
        assert torch.equal(caches[0], caches[2]) and torch.equal(caches[1], caches[3])


@pytest.mark.parametrize("tile", [5, 6])
@pytest.mark.parametrize("B,T,H,Hkv,hd,pos0,S", [(1, 193, 12, 12, 64, 0, 200), (3, 43, 4, 2, 128, 5, 60), (2, 97, 25, 25, 64, 9, 100)])
def test_qkv_scatter_tiles_between(tile, B, T, H, Hkv, hd, pos0, S):
    """The scatter epilogue of the tiles of 192 and 96 rows == qkv rows + qkv_split."""
    from distributed_neural_networks_amd.ops import gemm as G
    from distributed_neural_networks_amd.ops import transformer_ops as T_
    g = torch.Generator(device=DEV).manual_seed(B * T)
    d, N = 320, (H + 2 * Hkv) * hd
    x = torch.randn(B * T, d, device=DEV, generator=g).bfloat16()
    f = G.fold_norm(torch.randn(N, d, device=DEV, generator=g) * 0.05, torch.ones(d, device=DEV), torch.zeros(d, device=DEV),
                    torch.randn(N, device=DEV, generator=g) * 0.02, False, 1e-5, DEV)
    std, pos = torch.empty(B * T, d, device=DEV, dtype=torch.bfloat16), torch.full((B,), pos0, device=DEV, dtype=torch.int32)
    caches = [torch.zeros(B, Hkv, S, hd, device=DEV).bfloat16() for _ in range(4)]
    q, q2 = (torch.empty(B * H * T * hd, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    G.set_gemm_mid(tile)
    try:
        assert G.qkv_scatter_norm(x, f, std, q, caches[0], caches[1], pos, B, T, H, Hkv, hd)
        qkv = G.linear_norm(x, f, std_buf=std, ones=torch.ones(d, device=DEV))
    finally:
        G.set_gemm_mid()
    T_.qkv_split(qkv, q2, caches[2], caches[3], B, T, H, Hkv, hd, pos)
    keep = pos0 + torch.arange(T, device=DEV) < S
    assert torch.equal(q.view(B, H, T, hd)[:, :, keep], q2.view(B, H, T, hd)[:, :, keep])
    assert torch.equal(caches[0], caches[2]) and torch.equal(caches[1], caches[3])
