"""GPU tests of the NVFP4 recipe (TE 'nvfp4', bongard/te_linear.py:17,38; bongard/fused_mlp.py
:9,32) against the CPU oracle (oracle/fp8_oracle.py: quantize_nvfp4 and the chains built on it).

Quantization (codes, e4m3 block scales, meta) and the exact bf16 dequantization: bit-exact.
The bf16 MFMA GEMM: fp32 output within 1% of RMS of the fp64 product (measured ~1e-6), bf16
output the RNE of the fp32 output. A linear's forward and gradients on the same NVFP4 operands:
within 1% of RMS of the oracle's fp64 GEMMs (after half a bf16 ulp; measured 0 to 1.3e-7). The
gated MLP requantizes H (and dGU) into e2m1, where one bf16 ulp of g or u could move an H code
by a whole e2m1 step; the bf16 MFMA's sums of the exact block-dequantized products round to the
oracle's bf16 g and u here, so no code moves and the same 1% bar holds end to end (measured:
only the bf16 rounding of the outputs; the kernels are deterministic).
"""

import types

import pytest
import torch
from torch import nn
from transformers.models.t5gemma2.modeling_t5gemma2 import T5Gemma2MLP, T5Gemma2RMSNorm

from bongard_amd import fused_mlp, linear, ops, te_linear
from oracle import fp8_oracle as orc

pytestmark = pytest.mark.gpu


def _rms(t):
    return t.double().pow(2).mean().sqrt().item()


def _close(got, ref, what, tol=0.01):
    got, ref = got.float().cpu(), ref.float().cpu()
    excess = ((got - ref).abs() - 0.5 * orc.bf16_ulp(ref)).clamp(min=0).max().item()
    rel = excess / max(_rms(ref), 1e-30)
    print(f"[{what}] max(|err| - ulp/2)/RMS = {rel:.3e}", flush=True)
    assert rel <= tol, what


def _inputs(rows, cols, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(rows, cols, generator=g) * torch.rand(rows, 1, generator=g) * 4
    x[0, :16] = 0.0                              # an all-zero block
    x[1 % rows, 5] = 900.0                       # an outlier that sets the tensor scale
    x[2 % rows, 16:32] *= 1e-4                   # a block of small values
    return x.to(torch.bfloat16)


@pytest.mark.parametrize("rows,cols", [(64, 256), (48, 96), (300, 512), (16, 16)])
def test_quantize_nvfp4_bit_exact(gpu, rows, cols):
    x = _inputs(rows, cols, rows + cols)
    q = ops.quantize_nvfp4(x.to(gpu), rowwise=True, colwise=rows % 16 == 0)
    torch.cuda.synchronize()
    p, sb, s_enc, s_dec, a = orc.quantize_nvfp4(x)
    assert torch.equal(q.data.cpu(), p) and torch.equal(q.scales.cpu(), sb)
    assert q.meta.cpu().tolist() == [float(a), float(s_enc), float(s_dec), 0.0]
    if rows % 16 == 0:
        pt, st, _, _, _ = orc.quantize_nvfp4(x, axis=0)
        assert torch.equal(q.data_t.cpu(), pt) and torch.equal(q.scales_t.cpu(), st)
    deq = ops.dequant_nvfp4(q.data, q.scales)
    # the quantizer writing its rowwise copy as the bf16 dequantization directly
    qd = ops.quantize_nvfp4(x.to(gpu), rowwise=True, colwise=rows % 16 == 0, dequant_rows=True)
    torch.cuda.synchronize()
    assert qd.data is None and qd.scales is None
    assert torch.equal(ops.nvfp4_dequant(qd), deq) and torch.equal(qd.meta, q.meta)
    if rows % 16 == 0:
        assert torch.equal(qd.data_t, q.data_t) and torch.equal(qd.scales_t, q.scales_t)
    ref = orc.dequant_nvfp4(p, sb)
    assert torch.equal(deq.cpu().float(), ref)        # e2m1 x e4m3 is exact in bf16


@pytest.mark.parametrize("rows,cols", [(16, 128), (128, 128), (144, 272), (272, 48), (400, 2560),
                                       (1648, 2640)])
def test_quantize_nvfp4_tile_edges(gpu, rows, cols):
    """Whole and partial 128 x 128 tiles in either direction: codes and scales of both copies
    against the oracle, and both copies written as their bf16 dequantization."""
    x = _inputs(rows, cols, 7 * rows + cols)
    q = ops.quantize_nvfp4(x.to(gpu), rowwise=True, colwise=True)
    d = ops.quantize_nvfp4(x.to(gpu), rowwise=True, colwise=True, dequant_rows=True,
                           dequant_cols=True)
    dt = ops.quantize_nvfp4(x.to(gpu), rowwise=False, colwise=True, dequant_cols=True)
    torch.cuda.synchronize()
    p, sb, _, _, _ = orc.quantize_nvfp4(x)
    pt, st, _, _, _ = orc.quantize_nvfp4(x, axis=0)
    assert torch.equal(q.data.cpu(), p) and torch.equal(q.scales.cpu(), sb)
    assert torch.equal(q.data_t.cpu(), pt) and torch.equal(q.scales_t.cpu(), st)
    assert torch.equal(ops.nvfp4_dequant(d).cpu().float(), orc.dequant_nvfp4(p, sb))
    for t in (d, dt):
        assert t.data_t is None and torch.equal(t.meta, q.meta)
        assert torch.equal(ops.nvfp4_dequant(t, transpose=True).cpu().float(),
                           orc.dequant_nvfp4(pt, st))


@pytest.mark.parametrize("special", [None, float("inf"), float("nan")])
def test_quantize_nvfp4_broken_rows_and_non_finite(gpu, special):
    """Columns that do not fill 16-byte vectors: the same bytes as for those columns of a padded
    tensor under the same tensor amax, also where the tensor or some of its blocks hold inf or
    NaN."""
    x = _inputs(160, 24, 5)
    if special is not None:
        x[3, 4], x[100, 7] = special, -special
    x = x.to(gpu)
    parts = ops.amax(x)
    finite = ops.amax(torch.full((16, 8), 3.0, dtype=torch.bfloat16, device=gpu))
    for pr in (parts, finite):   # the tensor's own amax, and a finite scale for its blocks
        a = ops.quantize_nvfp4(x, rowwise=False, colwise=True, partials=pr)
        b = ops.quantize_nvfp4(x[:, :20].contiguous(), rowwise=False, colwise=True, partials=pr)
        torch.cuda.synchronize()
        assert torch.equal(a.data_t[:20], b.data_t) and torch.equal(a.scales_t[:20], b.scales_t)
    with pytest.raises(Exception, match="cols"):
        ops.quantize_nvfp4(x[:, :20].contiguous(), rowwise=False, colwise=True, dequant_cols=True)


@pytest.mark.parametrize("special", [None, float("inf"), float("nan")])
@pytest.mark.parametrize("rows", [16, 144, 1024])
def test_quantize_nvfp4_small_and_large_kernels(gpu, rows, special):
    """Tensors of up to 4M elements take kernels of their own: the first rows of a larger tensor
    quantized by themselves, under its amax, give the bytes that they have within it."""
    x = torch.randn(1040, 4096, generator=torch.Generator().manual_seed(rows)).to(torch.bfloat16)
    if special is not None:
        x[3, 4], x[rows - 1, 700] = special, -special
    x = x.to(gpu)
    assert x.numel() > 4 << 20 >= x[:rows].numel()
    for parts in (ops.amax(x), ops.amax(torch.full((16, 8), 3.0, dtype=torch.bfloat16, device=gpu))):
        big = ops.quantize_nvfp4(x, colwise=True, partials=parts)
        for args in (dict(), dict(dequant_rows=True), dict(rowwise=False)):
            small = ops.quantize_nvfp4(x[:rows], colwise=True, partials=parts, **args)
            torch.cuda.synchronize()
            if "dequant_rows" in args:
                want = ops.nvfp4_dequant(big)[:rows]
                assert torch.equal(ops.nvfp4_dequant(small).view(torch.int16), want.view(torch.int16))
            elif not args:
                assert torch.equal(small.data, big.data[:rows])
                assert torch.equal(small.scales, big.scales[:rows])
            assert torch.equal(small.data_t, big.data_t[:, :rows // 2])
            assert torch.equal(small.scales_t, big.scales_t[:, :rows // 16])
            assert torch.equal(small.meta.view(torch.int32), big.meta.view(torch.int32))


def test_quantize_nvfp4_zero_tensor_and_columnwise_only(gpu):
    x = torch.zeros(32, 64, dtype=torch.bfloat16)
    q = ops.quantize_nvfp4(x.to(gpu), rowwise=False, colwise=True)
    torch.cuda.synchronize()
    pt, st, s_enc, s_dec, _ = orc.quantize_nvfp4(x, axis=0)
    assert torch.equal(q.data_t.cpu(), pt) and torch.equal(q.scales_t.cpu(), st)
    assert q.meta.cpu().tolist() == [0.0, float(s_enc), float(s_dec), 0.0]
    assert int(q.data_t.count_nonzero()) == 0


@pytest.mark.parametrize("M,N,K", [(300, 328, 1040), (4096, 2560, 2560), (512, 2560, 10240)])
def test_gemm_bf16(gpu, M, N, K):
    g = torch.Generator().manual_seed(M + N)
    a = torch.randn(M, K, generator=g).to(torch.bfloat16)
    b = (torch.randn(N, K, generator=g) * 0.02).to(torch.bfloat16)
    sa = torch.tensor([0.5], device=gpu)
    sb = torch.tensor([3.0], device=gpu)
    y32 = ops.gemm_bf16(a.to(gpu), b.to(gpu), sa, sb, out_dtype=torch.float32)
    y16 = ops.gemm_bf16(a.to(gpu), b.to(gpu), sa, sb)
    torch.cuda.synchronize()
    rows = torch.arange(0, M, max(1, M // 128))
    ref = (a[rows].double() @ b.double().t()) * 1.5
    err = (y32.cpu()[rows].double() - ref).abs().max().item() / _rms(ref)
    print(f"[gemm_bf16 {M}x{N}x{K}] max|err|/RMS = {err:.3e}", flush=True)
    assert err <= 0.01
    assert torch.equal(y16.cpu().view(torch.int16), y32.cpu().to(torch.bfloat16).view(torch.int16))


@pytest.mark.parametrize("tile", ["256x256w8", "256x256w8x", "256x160", "128x64k2"])
def test_gemm_bf16_tiles(gpu, monkeypatch, tile):
    """The bf16 operand format on forced tiles (the eight-wave tile with and without its third
    B slot among them), with M, N and K tails: the fp32 output against the fp64 product."""
    monkeypatch.setenv("BONGARD_FP8_GEMM_TILE", tile)
    g = torch.Generator().manual_seed(71)
    M, N, K = 300, 328, 1040  # 2080 bytes of K: 16 whole 128-byte steps and a partial one
    a = torch.randn(M, K, generator=g).to(torch.bfloat16)
    b = (torch.randn(N, K, generator=g) * 0.02).to(torch.bfloat16)
    one = torch.tensor([1.0], device=gpu)
    y = ops.gemm_bf16(a.to(gpu), b.to(gpu), one, one, out_dtype=torch.float32)
    torch.cuda.synchronize()
    ref = a.double() @ b.double().t()
    err = (y.cpu().double() - ref).abs().max().item() / _rms(ref)
    print(f"[gemm_bf16 {tile}] max|err|/RMS = {err:.3e}", flush=True)
    assert err <= 0.01


def test_gemm_nvfp4_on_own_operands(gpu):
    x = _inputs(256, 512, 3)
    w = (torch.randn(384, 512, generator=torch.Generator().manual_seed(4)) * 0.02).to(torch.bfloat16)
    xq, wq = ops.quantize_nvfp4(x.to(gpu)), ops.quantize_nvfp4(w.to(gpu))
    y = ops.gemm_nvfp4(xq.data, xq.scales, xq.meta, wq.data, wq.scales, wq.meta,
                       out_dtype=torch.float32)
    torch.cuda.synchronize()
    px, sx, _, dx, _ = orc.quantize_nvfp4(x)
    pw, sw, _, dw, _ = orc.quantize_nvfp4(w)
    _close(y, orc.scaled_mm_nvfp4(px, sx, dx, pw, sw, dw), "nvfp4 GEMM")


@pytest.mark.parametrize("rows", [512, 300])
def test_telinear_nvfp4_fwd_bwd(gpu, rows):
    """The linear's forward and both gradients on bit-exact NVFP4 operands: the 1% bar."""
    g = torch.Generator().manual_seed(rows)
    x = torch.randn(rows, 512, generator=g).to(torch.bfloat16)
    w = (torch.randn(384, 512, generator=g) * 0.02).to(torch.bfloat16)
    dy = (torch.randn(rows, 384, generator=g) * 1e-3).to(torch.bfloat16)
    lin = nn.Linear(512, 384, bias=False)
    lin.weight.data = w.clone().float()
    t = te_linear.TELinear([lin], "nvfp4").to(gpu).train()
    xg = x.to(gpu).requires_grad_(True)
    y = t(xg)
    y.backward(dy.to(gpu))
    torch.cuda.synchronize()
    pad = (rows + 31) // 32 * 32 - rows
    ry, rdx, rdw = orc.linear_fwd_bwd_nvfp4(torch.nn.functional.pad(x, (0, 0, 0, pad)), w,
                                            torch.nn.functional.pad(dy, (0, 0, 0, pad)))
    _close(y, ry[:rows], "nvfp4 linear y")
    _close(xg.grad, rdx[:rows], "nvfp4 linear dx")
    _close(t.weight.grad, rdw, "nvfp4 linear dW")
    assert t.counts == {"weight_quantizations": 1}
    t(xg)
    assert t.counts == {"weight_quantizations": 1, "cached_weights": 1}


@pytest.mark.parametrize("rows,K,I", [(512, 256, 512), (304, 512, 384), (64, 128, 256)])
def test_geglu_gate_up_nvfp4_equals_unfused(gpu, rows, K, I):
    """The gate/up GEMM with the gated GELU in its bf16 epilogue (bf8_gemm_geglu_bf16)
    against the unfused chain on the same inputs (the NVFP4 linear, then the elementwise
    gated GELU): H, and both gradients from the same dH, bit for bit (the GEMM plans here
    run unsplit, so both sum every output in the same order); H also within the 1% bar of
    the oracle's chain, and the no-grad forward (which keeps no GU) equal to the training
    one."""
    g = torch.Generator().manual_seed(rows + K + I)
    x = _inputs(rows, K, rows + K)
    w = (torch.randn(2 * I, K, generator=g) * 0.02).to(torch.bfloat16)
    dH = (torch.randn(rows, I, generator=g) * 1e-3).to(torch.bfloat16).to(gpu)
    x1, w1 = x.to(gpu).requires_grad_(True), w.to(gpu).requires_grad_(True)
    H1, hp1 = linear.GegluGateUpNvfp4Function.apply(x1, w1, None, I)
    H1.backward(dH)
    x2, w2 = x.to(gpu).requires_grad_(True), w.to(gpu).requires_grad_(True)
    H2, hp2 = linear.GegluFunction.apply(linear.Fp8LinearNvfp4Function.apply(x2, w2, None))
    H2.backward(dH)
    with torch.no_grad():
        H0, _ = linear.GegluGateUpNvfp4Function.apply(x.to(gpu), w.to(gpu), None, I)
    torch.cuda.synchronize()
    assert H1.shape == (rows, I)
    assert torch.equal(H1, H2), "H"
    assert torch.equal(H0, H1), "H without grad"
    assert torch.equal(x1.grad, x2.grad), "dx"
    assert torch.equal(w1.grad, w2.grad), "dW"
    assert not hp1.requires_grad
    assert hp1.max().item() == H2.abs().float().max().view(torch.int32).item(), "H partials"
    assert hp2.max().item() == hp1.max().item() and not hp2.requires_grad
    # a weight cached across microbatches keeps its bf16 dequantizations: the first call
    # fills them, the second reads them; both equal the uncached path bit for bit
    wq = linear.quantize_weight_nvfp4(w.to(gpu), cache_dequant=True)
    for call in range(2):
        x3, w3 = x.to(gpu).requires_grad_(True), w.to(gpu).requires_grad_(True)
        H3, _ = linear.GegluGateUpNvfp4Function.apply(x3, w3, wq, I)
        H3.backward(dH)
        y3 = linear.Fp8LinearNvfp4Function.apply(x3.detach().requires_grad_(True), w3, wq)
        torch.cuda.synchronize()
        assert wq._deq is not None and wq._deq_t is not None, call
        assert torch.equal(H3, H1) and torch.equal(x3.grad, x1.grad), call
        assert torch.equal(w3.grad, w1.grad), call
        y4 = linear.Fp8LinearNvfp4Function.apply(x.to(gpu), w.to(gpu), None)
        assert torch.equal(y3, y4), call
    gu = orc.linear_fwd_bwd_nvfp4(x, w, torch.zeros(rows, 2 * I, dtype=torch.bfloat16))[0]
    _close(H1, orc.geglu(gu[:, :I].to(torch.bfloat16), gu[:, I:].to(torch.bfloat16)),
           "nvfp4 fused gate/up H")


@pytest.mark.parametrize("rows", [96, 80])
def test_quantize_nvfp4_from_producer_partials(gpu, rows):
    """The NVFP4 quantizer fed the amax partials its producer wrote (geglu_bwd's for dGU,
    the gated-GELU GEMM's epilogue for H, the fused RMSNorm's for its output) against its
    own amax pass: codes, block scales (both directions) and meta bit for bit. rows = 80 is
    not a whole number of GEMM tiles (the rows past M must add nothing to H's partials)."""
    g = torch.Generator().manual_seed(rows)
    I, K = 256, 128
    GU = (torch.randn(rows, 2 * I, generator=g) * 2).to(torch.bfloat16).to(gpu)
    dH = (torch.randn(rows, I, generator=g) * 1e-3).to(torch.bfloat16).to(gpu)
    x = _inputs(rows, K, rows + 1).to(gpu)
    w = (torch.randn(2 * I, K, generator=g) * 0.02).to(torch.bfloat16).to(gpu)
    gamma = (torch.randn(K, generator=g) * 0.1).to(torch.bfloat16).to(gpu)
    dGU, dparts = ops.geglu_bwd(dH, GU)
    xq, wq = ops.quantize_nvfp4(x), ops.quantize_nvfp4(w)
    H, _, hparts = ops.gemm_geglu_nvfp4(xq.data, xq.scales, xq.meta, wq.data, wq.scales,
                                        wq.meta, I)
    normed, _, nparts = ops.rmsnorm(x, gamma, 1e-6)
    for what, t, parts in (("dGU", dGU, dparts), ("H", H, hparts), ("normed", normed, nparts)):
        for rw, cw in ((True, True), (True, False), (False, True)):
            a = ops.quantize_nvfp4(t, rowwise=rw, colwise=cw)
            b = ops.quantize_nvfp4(t, rowwise=rw, colwise=cw, partials=parts)
            torch.cuda.synchronize()
            for f in ("data", "scales", "data_t", "scales_t"):
                fa, fb = getattr(a, f), getattr(b, f)
                assert (fa is None) == (fb is None), (what, f)
                assert fa is None or torch.equal(fa, fb), (what, rw, cw, f)
            assert torch.equal(a.meta, b.meta), (what, rw, cw, "meta")
            if rw:
                c = ops.quantize_nvfp4(t, rowwise=True, colwise=cw, partials=parts,
                                       dequant_rows=True)
                torch.cuda.synchronize()
                assert torch.equal(ops.nvfp4_dequant(c), ops.dequant_nvfp4(a.data, a.scales))
                assert torch.equal(c.meta, a.meta) and (not cw or torch.equal(c.data_t, a.data_t))
    with pytest.raises(ValueError):
        ops.quantize_nvfp4(H, partials=hparts.float())


def _mlp(hidden, inter, seed):
    cfg = types.SimpleNamespace(hidden_size=hidden, intermediate_size=inter,
                                hidden_activation="gelu_pytorch_tanh", dropout_rate=0.0)
    torch.manual_seed(seed)
    m = T5Gemma2MLP(cfg)
    with torch.no_grad():
        m.gate_proj.weight.normal_(std=0.02)
        m.up_proj.weight.normal_(std=0.02)
        m.down_proj.weight.normal_(std=0.014)
    return m.to(torch.bfloat16)


@pytest.mark.parametrize("split", [False, True])
def test_temlp_nvfp4_fwd_bwd(gpu, monkeypatch, split):
    """TEMLP under 'nvfp4' (fused gate_up, or BONGARD_TE_SPLIT_GATE_UP=1 with one tensor
    scale per projection) against the oracle's NVFP4 chain: H and dGU are requantized to
    e2m1 inside, so the bar is statistical."""
    if split:
        monkeypatch.setenv("BONGARD_TE_SPLIT_GATE_UP", "1")
    g = torch.Generator().manual_seed(61)
    rows, hidden, I = 512, 256, 512
    mlp = _mlp(hidden, I, 61)
    wg, wu, wd = (m.weight.detach().clone() for m in (mlp.gate_proj, mlp.up_proj, mlp.down_proj))
    x = torch.randn(rows, hidden, generator=g).to(torch.bfloat16)
    dy = (torch.randn(rows, hidden, generator=g) * 1e-3).to(torch.bfloat16)
    t = te_linear.TEMLP(mlp, "nvfp4").to(gpu).train()
    assert t.fused_gate_up != split
    xg = x.to(gpu).requires_grad_(True)
    y = t(xg)
    y.backward(dy.to(gpu))
    torch.cuda.synchronize()
    if split:
        gq = orc.linear_fwd_bwd_nvfp4(x, wg, torch.zeros(rows, I, dtype=torch.bfloat16))[0]
        uq = orc.linear_fwd_bwd_nvfp4(x, wu, torch.zeros(rows, I, dtype=torch.bfloat16))[0]
        h = orc.geglu(gq.to(torch.bfloat16), uq.to(torch.bfloat16))
        ry = orc.linear_fwd_bwd_nvfp4(h, wd, dy)[0]
        _close(y, ry, "nvfp4 split y")
        assert t.gate_proj.weight.grad is not None and t.up_proj.weight.grad is not None
        return
    ry, rdx, rdwgu, rdwd = orc.mlp_fwd_bwd_nvfp4(x, wg, wu, wd, dy)
    _close(y, ry, "nvfp4 temlp y")
    _close(xg.grad, rdx, "nvfp4 temlp dx")
    _close(t.gate_up.weight.grad, rdwgu, "nvfp4 temlp dWgu")
    _close(t.down.weight.grad, rdwd, "nvfp4 temlp dWd")


def test_fused_mlp_nvfp4_fwd_bwd(gpu):
    g = torch.Generator().manual_seed(62)
    rows, hidden, I = 256, 256, 512
    mlp = _mlp(hidden, I, 62)
    norm = T5Gemma2RMSNorm(hidden, eps=1e-6).to(torch.bfloat16)
    with torch.no_grad():
        norm.weight.normal_(std=0.1)
    wg, wu, wd = (m.weight.detach().clone() for m in (mlp.gate_proj, mlp.up_proj, mlp.down_proj))
    nw = norm.weight.detach().clone()
    x = torch.randn(rows, hidden, generator=g).to(torch.bfloat16)
    dy = (torch.randn(rows, hidden, generator=g) * 1e-3).to(torch.bfloat16)
    f = fused_mlp.FusedMLP(mlp, norm, "nvfp4").to(gpu).train()
    xg = x.to(gpu).requires_grad_(True)
    y = f(xg)
    y.backward(dy.to(gpu))
    torch.cuda.synchronize()
    normed = orc.rmsnorm(x, nw, 1e-6)
    ry, _, rdwgu, rdwd = orc.mlp_fwd_bwd_nvfp4(normed, wg, wu, wd, dy)
    _close(y, ry, "nvfp4 fused y")
    _close(f.fc1_weight.grad, rdwgu, "nvfp4 fused dW_fc1")
    _close(f.fc2_weight.grad, rdwd, "nvfp4 fused dW_fc2")
    assert xg.grad is not None and f.layer_norm_weight.grad is not None
    assert f.state_dict()["_extra_state"].numel() == 0
