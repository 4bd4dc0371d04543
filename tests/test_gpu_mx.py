"""GPU parity of the MXFP8 path (TE MXFP8BlockScaling arithmetic) against the CPU oracle.

  * quantize: fp8 bytes and E8M0 scale rows (padding bytes included) bit-exact against
    oracle.quantize_mx, blocks along rows and (transposed) along columns;
  * block-scaled GEMM: fp32 output within 1% of RMS of the oracle's fp64 dequantized
    matmul, bf16 output the RNE rounding of the same kernel's fp32 output;
  * gated-GELU GEMM on MX operands: bf16 pre-activations within 0.1% RMS (after half an
    ulp) of the fp64 GEMMs, and H within 2 bf16 ulps of the gelu chain on its own g, u.
"""

import pytest
import torch

from bongard_amd import ops
from oracle import fp8_oracle as orc

pytestmark = pytest.mark.gpu


def _rms(t):
    return t.double().pow(2).mean().sqrt().item()


def _x(rows, cols, seed, spread=True):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(rows, cols, generator=g)
    if spread and rows >= 8 and cols >= 64:
        x *= torch.logspace(-6, 6, rows)[:, None]       # many binades across rows
        x[:, 5] *= 300.0                                 # an outlier column
        x[3, 32:64] = 0.0                                # an all-zero block
    return x.to(torch.bfloat16)


@pytest.mark.parametrize("rows,cols", [(32, 32), (64, 2560), (96, 4096), (4096, 2560),
                                       (160, 10240), (32, 48)])
@pytest.mark.parametrize("fmt", [ops.E4M3, ops.E5M2])
def test_quantize_mx_bit_exact(gpu, rows, cols, fmt):
    x = _x(rows, cols, rows + cols + fmt)
    rowwise = cols % 32 == 0
    q = ops.quantize_mx(x.to(gpu), fmt, rowwise=rowwise, colwise=True)
    torch.cuda.synchronize()
    if rowwise:
        rq, re = orc.quantize_mx(x, fmt, -1)
        same_q = torch.equal(q.data.view(torch.uint8).cpu(), rq)
        same_s = torch.equal(q.scales.cpu(), orc.mx_scale_rows(re))
        print(f"[mx rows {rows}x{cols} fmt {fmt}] bytes {same_q} scales {same_s}", flush=True)
        assert same_q and same_s
    cq, ce = orc.quantize_mx(x, fmt, 0)
    same_q = torch.equal(q.data_t.view(torch.uint8).cpu(), cq)
    same_s = torch.equal(q.scales_t.cpu(), orc.mx_scale_rows(ce))
    print(f"[mx cols {rows}x{cols} fmt {fmt}] bytes {same_q} scales {same_s}", flush=True)
    assert same_q and same_s


@pytest.mark.parametrize("rows,cols", [(32, 32), (128, 128), (160, 96), (288, 416), (64, 144),
                                       (4128, 2144), (8352, 1040)])
def test_quantize_mx_two_copies_edges(gpu, rows, cols):
    """Both copies from one pass over 32 x 64 tiles (small tensors) and 128 x 128 tiles (the last
    two, past 8 x 2^20 elements): whole and partial tiles in either direction (scale padding
    included), both layouts of the scales, blocks holding inf, NaN and the largest and smallest
    magnitudes, and the columnwise copy alone."""
    x = _x(rows, cols, 3 * rows + cols, spread=False).float()
    x[1, 3], x[rows - 1, cols - 1], x[rows // 2, cols // 2] = float("inf"), float("nan"), -float("inf")
    x[2, :16] = 3.38e38
    x[3, 16:32] = 1e-39
    x = x.to(torch.bfloat16)
    rowwise = cols % 32 == 0
    q = ops.quantize_mx(x.to(gpu), rowwise=rowwise, colwise=True)
    only = ops.quantize_mx(x.to(gpu), rowwise=False, colwise=True)
    torch.cuda.synchronize()
    cq, ce = orc.quantize_mx(x, ops.E4M3, 0)
    for t in (q, only):
        assert torch.equal(t.data_t.view(torch.uint8).cpu(), cq)
        assert torch.equal(t.scales_t.cpu(), orc.mx_scale_rows(ce))
        assert torch.equal(t.planes_t, _planes_of(t.scales_t))
    if rowwise:
        rq, re = orc.quantize_mx(x, ops.E4M3, -1)
        assert torch.equal(q.data.view(torch.uint8).cpu(), rq)
        assert torch.equal(q.scales.cpu(), orc.mx_scale_rows(re))
        assert torch.equal(q.planes, _planes_of(q.scales))


def test_quantize_mx_errors(gpu):
    with pytest.raises(Exception, match="cols"):
        ops.quantize_mx(torch.zeros(32, 48, dtype=torch.bfloat16, device=gpu))
    with pytest.raises(Exception, match="rows"):
        ops.quantize_mx(torch.zeros(48, 64, dtype=torch.bfloat16, device=gpu), colwise=True)


@pytest.mark.parametrize("rows,cols", [(1, 32), (3, 96), (33, 128), (95, 160), (128, 416), (300, 1056),
                                       (3001, 2112)])
def test_quantize_mx_rows_alone(gpu, rows, cols):
    """The rowwise copy alone: rows and columns that leave partial wave tiles of 4 x 128 (small
    tensors) and 16 x 128 (the last, past 6 x 2^20 elements), with and without inf, NaN and the
    largest and smallest magnitudes; bytes and both layouts of the scales, one tensor or several,
    against the oracle."""
    x = _x(rows, cols, rows + cols, spread=False)
    y = x.float()
    y[0, :16], y[rows - 1, 16:32] = 3.38e38, 1e-39
    y[rows // 2, cols - 1], y[rows - 1, 3] = float("nan"), -float("inf")
    xs = [x, y.to(torch.bfloat16)]
    for fmt in (ops.E4M3, ops.E5M2):
        many = ops.quantize_mx_many([t.to(gpu) for t in xs], fmt)
        for t, m in zip(xs, many):
            rq, re = orc.quantize_mx(t, fmt, -1)
            for q in (ops.quantize_mx(t.to(gpu), fmt), m):
                assert torch.equal(q.data.view(torch.uint8).cpu(), rq)
                assert torch.equal(q.scales.cpu(), orc.mx_scale_rows(re))
                assert torch.equal(q.planes, _planes_of(q.scales))
            alone = ops.quantize_mx(t.to(gpu), fmt, scale_rows=False)
            assert torch.equal(alone.data.view(torch.uint8), m.data.view(torch.uint8))
            assert torch.equal(alone.planes, m.planes)


def _planes_of(rows_scales):
    """The scale planes [ld / 4, rows] of scale rows [rows, ld]."""
    r, ld = rows_scales.shape
    return rows_scales.contiguous().view(torch.int32).reshape(r, ld // 4).t().contiguous()


@pytest.mark.parametrize("rows,cols", [(32, 32), (160, 96), (288, 416), (512, 2560)])
def test_mx_scale_planes(gpu, rows, cols):
    """The quantizers' scale planes hold the scale rows' dwords (either copy, one tensor or
    several), and a GEMM on planes gives the bits of the GEMM on rows."""
    x = _x(rows, cols, rows - cols).to(gpu)
    w = _x(64, cols, cols, spread=False).to(gpu)
    q, qw = ops.quantize_mx(x, colwise=True), ops.quantize_mx(w)
    many = ops.quantize_mx_many([x, w])
    assert torch.equal(q.planes, _planes_of(q.scales))
    assert torch.equal(q.planes_t, _planes_of(q.scales_t))
    for a, b in zip(many, (q, qw)):
        assert torch.equal(a.planes, b.planes) and torch.equal(a.scales, b.scales)
    y = ops.gemm_mx(q.data, q.scales, qw.data, qw.scales)
    yp = ops.gemm_mx(q.data, None, qw.data, None, a_planes=q.planes, b_planes=qw.planes)
    assert torch.equal(y, yp)
    with pytest.raises(ValueError, match="a_planes"):
        ops.gemm_mx(q.data, None, qw.data, None, a_planes=qw.planes, b_planes=q.planes)


@pytest.mark.parametrize("tile", ["", "256x256w8"])
@pytest.mark.parametrize("M,I,K", [(32, 128, 96), (288, 384, 512), (512, 1280, 2560)])
def test_gemm_geglu_mx_planes(gpu, monkeypatch, tile, M, I, K):
    """The gated-GELU GEMM on planes: H's bytes, its planes (both copies) and GU equal those of
    the GEMM on scale rows (which test_gemm_geglu_mx_quant holds against the oracle)."""
    monkeypatch.setenv("BONGARD_FP8_GEMM_TILE", tile)
    x = _x(M, K, M, spread=False).to(gpu)
    w = (_x(2 * I, K, I, spread=False).float() * 0.02).to(torch.bfloat16).to(gpu)
    qx, qw = ops.quantize_mx(x), ops.quantize_mx(w)
    hq, gu, _ = ops.gemm_geglu_mx_quant(qx.data, qx.scales, qw.data, qw.scales, I, colwise=True,
                                        keep_gu=True)
    hp, gup = ops.gemm_geglu_mx_planes(qx.data, qx.planes, qw.data, qw.planes, I, colwise=True,
                                       keep_gu=True)
    u8 = torch.uint8
    assert torch.equal(hq.data.view(u8), hp.data.view(u8)) and torch.equal(gu, gup)
    assert torch.equal(hq.data_t.view(u8), hp.data_t.view(u8))
    ld = ops.mx_scale_ld(I)
    assert torch.equal(_planes_of(hq.scales[:, :ld]), hp.planes)
    assert torch.equal(_planes_of(hq.scales_t), hp.planes_t)


def _mx_gemm_case(gpu, M, N, K, seed, bias=False):
    g = torch.Generator().manual_seed(seed)
    a = (torch.randn(M, K, generator=g) * torch.logspace(-2, 2, K)[None, :]).to(torch.bfloat16)
    b = (torch.randn(N, K, generator=g) * 0.02).to(torch.bfloat16)
    bias_t = (torch.randn(N, generator=g) * 0.1).to(torch.bfloat16) if bias else None
    qa = ops.quantize_mx(a.to(gpu))
    qb = ops.quantize_mx(b.to(gpu))
    bias_g = bias_t.to(gpu) if bias else None
    y32 = ops.gemm_mx(qa.data, qa.scales, qb.data, qb.scales, out_dtype=torch.float32, bias=bias_g)
    y16 = ops.gemm_mx(qa.data, qa.scales, qb.data, qb.scales, bias=bias_g)
    planes = ops.gemm_mx(qa.data, None, qb.data, None, a_planes=qa.planes, b_planes=qb.planes,
                         bias=bias_g)
    torch.cuda.synchronize()
    assert torch.equal(planes.view(torch.int16), y16.view(torch.int16))
    ra, ea = orc.quantize_mx(a, ops.E4M3)
    rb, eb = orc.quantize_mx(b, ops.E4M3)
    assert torch.equal(qa.data.view(torch.uint8).cpu(), ra)
    assert torch.equal(qb.data.view(torch.uint8).cpu(), rb)
    ref = orc.scaled_mm_mx(ra, ea, rb, eb, bias=bias_t)
    err = (y32.cpu() - ref).abs().max().item() / max(_rms(ref), 1e-30)
    print(f"[mx gemm {M}x{N}x{K}] max|err|/RMS = {err:.3e}", flush=True)
    assert err <= 0.01
    assert torch.equal(y16.cpu().view(torch.int16), y32.cpu().to(torch.bfloat16).view(torch.int16))


@pytest.mark.parametrize("M,N,K", [
    (512, 2048, 2560),     # c1 shape
    (100, 264, 352),       # ragged M, N; K % 128 = 96 (a partial last K step)
    (4096, 2560, 2560),    # large tiles
    (512, 2560, 10240),    # split-K (partials reduced with unit scale)
    (64, 128, 32),         # a single block of K
])
def test_gemm_mx(gpu, M, N, K):
    _mx_gemm_case(gpu, M, N, K, seed=M + N + K)


def test_gemm_mx_bias(gpu):
    _mx_gemm_case(gpu, 200, 256, 512, seed=5, bias=True)


@pytest.mark.parametrize("tile", ["256x256", "256x256w8"])
def test_gemm_mx_tail_split(gpu, monkeypatch, tile):
    """MX operands under the tail split (272 tiles of 256x256, 16 of them split along K):
    the tail tiles' pieces are reduced with unit scales."""
    monkeypatch.setenv("BONGARD_FP8_GEMM_TILE", tile + ":t")
    M, N, K = 4160, 3848, 4096
    assert ops._lib.lib().bf8_gemm_mx_workspace(M, N, K) % (16 * 256 * 256 * 4) == 0
    _mx_gemm_case(gpu, M, N, K, seed=63, bias=True)


@pytest.mark.parametrize("M,I,K", [(300, 384, 512), (512, 1024, 2560), (64, 128, 96)])
def test_gemm_geglu_mx(gpu, M, I, K):
    g = torch.Generator().manual_seed(M + I)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16)
    w = (torch.randn(2 * I, K, generator=g) * 0.02).to(torch.bfloat16)
    qx = ops.quantize_mx(x.to(gpu))
    qw = ops.quantize_mx(w.to(gpu))
    H, GU = ops.gemm_geglu_mx(qx.data, qx.scales, qw.data, qw.scales, I, keep_gu=True)
    torch.cuda.synchronize()
    rx, ex = orc.quantize_mx(x, ops.E4M3)
    rw, ew = orc.quantize_mx(w, ops.E4M3)
    gate = orc.scaled_mm_mx(rx, ex, rw[:I], ew[:I])
    up = orc.scaled_mm_mx(rx, ex, rw[I:], ew[I:])
    GU_c, H_c = GU.cpu(), H.cpu()
    for got, ref, what in ((GU_c[:, :I], gate, "gate"), (GU_c[:, I:], up, "up")):
        excess = ((got.float() - ref).abs() - 0.5 * orc.bf16_ulp(ref)).max().item()
        rel = excess / max(_rms(ref), 1e-30)
        print(f"[mx geglu {what} {M}x{I}x{K}] max(|err| - ulp/2)/RMS = {rel:.3e}", flush=True)
        assert rel <= 1e-3
    H_ref = orc.geglu(GU_c[:, :I], GU_c[:, I:])
    diff = (H_c.float() - H_ref.float()).abs()
    ulp = orc.bf16_ulp(H_ref.float())
    slack = 2.0 ** -20 * H_ref.float().abs().max()
    assert bool((diff <= 2 * ulp + slack).all()), "H beyond 2 bf16 ulps of the gelu chain"
    assert (diff > 0).float().mean().item() <= 0.05


GEGLU_TILES = ["256x256", "160x256", "192x256", "128x128", "64x128", "256x128", "256x256w8"]


@pytest.mark.parametrize("tile", ["auto"] + GEGLU_TILES)
@pytest.mark.parametrize("M,I,K", [(320, 384, 256), (100, 256, 128), (288, 128, 352), (33, 128, 512)])
def test_gemm_geglu_mx_quant(gpu, monkeypatch, tile, M, I, K):
    """H quantized in the GEGLU epilogue == bf8_quantize_mx_bf16 of the bf16 H of the
    unfused kernel, byte for byte (fp8 payloads, E8M0 scales, the transposed copy and its
    padding), on every tile with a gated-GELU variant, with inf / NaN blocks in H."""
    if tile != "auto":
        monkeypatch.setenv("BONGARD_FP8_GEMM_TILE", tile)
    g = torch.Generator().manual_seed(M + I + K)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16)
    x[7] *= 1e-4                      # a row of small activations
    w = (torch.randn(2 * I, K, generator=g) * 0.02).to(torch.bfloat16)
    qx = ops.quantize_mx(x.to(gpu))
    qw = ops.quantize_mx(w.to(gpu))
    qx.scales[5, 0] = 254             # row 5: 2^127 on its first block -> +-inf gate/up, NaN H
    qx.data.view(torch.uint8)[9, 3] = 0x7F  # row 9: an e4m3 NaN operand -> NaN row of H
    colwise = M % 32 == 0
    args = (qx.data, qx.scales, qw.data, qw.scales, I)
    hq, GU, H = ops.gemm_geglu_mx_quant(*args, colwise=colwise, keep_gu=True, keep_h=True)
    hq2, GU2, H2 = ops.gemm_geglu_mx_quant(*args, colwise=colwise)
    H_ref, GU_ref = ops.gemm_geglu_mx(*args, keep_gu=True)
    ref = ops.quantize_mx(H_ref, rowwise=True, colwise=colwise)
    torch.cuda.synchronize()
    assert GU2 is None and H2 is None and (hq2.data_t is None) == (not colwise)
    assert torch.equal(H.view(torch.int16), H_ref.view(torch.int16))
    assert torch.equal(GU.view(torch.int16), GU_ref.view(torch.int16))
    hc = H_ref.cpu()
    assert bool(hc[9].isnan().any()) and bool(hc[5].isinf().any() or hc[5].isnan().any())
    for q, what in ((hq, "with H"), (hq2, "without H")):
        same = [torch.equal(q.data.view(torch.uint8), ref.data.view(torch.uint8)),
                torch.equal(q.scales, ref.scales)]
        if colwise:
            same += [torch.equal(q.data_t.view(torch.uint8), ref.data_t.view(torch.uint8)),
                     torch.equal(q.scales_t, ref.scales_t)]
        print(f"[mx geglu quant {tile} {M}x{I}x{K} {what}] rows, scales, cols, scales_t: "
              f"{same}", flush=True)
        assert all(same)
    # and the oracle on the finite rows (the kernel's own H as input)
    finite = hc.isfinite().all(dim=1)
    rq, re_ = orc.quantize_mx(hc[finite], ops.E4M3)
    assert torch.equal(hq.data.view(torch.uint8).cpu()[finite], rq)
    assert torch.equal(hq.scales.cpu()[finite][:, :I // 32], re_.to(torch.uint8))


def test_gemm_geglu_mx_quant_errors(gpu):
    qx = ops.quantize_mx(torch.randn(100, 128, device=gpu).to(torch.bfloat16))
    qw = ops.quantize_mx(torch.randn(512, 128, device=gpu).to(torch.bfloat16))
    with pytest.raises(RuntimeError, match="M % 32"):
        ops.gemm_geglu_mx_quant(qx.data, qx.scales, qw.data, qw.scales, 256, colwise=True)


@pytest.mark.parametrize("M,I,rowwise,colwise", [
    (M, I, *copies) for M, I in [(32, 128), (96, 384), (128, 256), (160, 128), (1056, 640),
                                 (2080, 1536), (4128, 1536)]
    for copies in [(True, True), (True, False), (False, True)]] + [
    (M, I, True, False) for M, I in [(1, 128), (45, 256), (4131, 1536)]])
def test_geglu_bwd_mx_equals_two_passes(gpu, M, I, rowwise, colwise):
    """The fused gated-GELU backward and MX quantizer, by wave tiles of 32 x 64 and, past 6 x 2^20
    elements of dGU (12 x 2^20 rowwise alone), tiles of 128 x 128: odd tile counts, partial tile
    rows, an inf and a NaN gradient, against geglu_bwd and quantize_mx: the
    same bytes and scale planes."""
    g = torch.Generator().manual_seed(M + I)
    dH = torch.randn(M, I, generator=g)
    dH[M - 1, I - 1], dH[M // 2, 5] = float("inf"), float("nan")
    GU = 3 * torch.randn(M, 2 * I, generator=g)
    dH, GU = dH.bfloat16().to(gpu), GU.bfloat16().to(gpu)
    one = ops.geglu_bwd_mx(dH, GU, rowwise=rowwise, colwise=colwise)
    two = ops.quantize_mx(ops.geglu_bwd(dH, GU)[0], rowwise=rowwise, colwise=colwise,
                          scale_rows=False)
    torch.cuda.synchronize()
    for a, b in ((one.data, two.data), (one.planes, two.planes), (one.data_t, two.data_t),
                 (one.planes_t, two.planes_t)):
        assert (a is None) == (b is None)
        assert a is None or torch.equal(a.view(torch.uint8), b.view(torch.uint8))


# ---- the TE modules under 'mxfp8' ------------------------------------------------------
import types  # noqa: E402

from torch import nn  # noqa: E402
from transformers.models.t5gemma2.modeling_t5gemma2 import T5Gemma2MLP, T5Gemma2RMSNorm  # noqa: E402

from bongard_amd import fused_mlp, te_linear  # noqa: E402


def _close(got, ref, what, tol=0.01):
    got, ref = got.float().cpu(), ref.float().cpu()
    excess = ((got - ref).abs() - 0.5 * orc.bf16_ulp(ref)).clamp(min=0).max().item()
    rel = excess / max(_rms(ref), 1e-30)
    print(f"[{what}] max(|err| - ulp/2)/RMS = {rel:.3e}", flush=True)
    assert rel <= tol, what


def _close_requant(got, ref, what, max_tol=0.05, rms_tol=0.005):
    """H (and dGU) are requantized inside the chain: sparse legitimate fp8 flips where
    GPU and oracle round a value to neighbouring bf16s; statistical bar as for 'fp8'."""
    got, ref = got.float().cpu(), ref.float().cpu()
    rms = max(_rms(ref), 1e-30)
    max_rel = (got - ref).abs().max().item() / rms
    rms_rel = _rms(got - ref) / rms
    print(f"[{what}] max|err|/RMS = {max_rel:.3e}, RMS(err)/RMS = {rms_rel:.3e}", flush=True)
    assert max_rel <= max_tol and rms_rel <= rms_tol, what


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


@pytest.mark.parametrize("rows", [256, 200])
def test_telinear_mxfp8_fwd_bwd(gpu, rows):
    g = torch.Generator().manual_seed(rows + 1)
    x = torch.randn(rows, 512, generator=g).to(torch.bfloat16)
    w = (torch.randn(384, 512, generator=g) * 0.02).to(torch.bfloat16)
    dy = (torch.randn(rows, 384, generator=g) * 1e-3).to(torch.bfloat16)
    lin = nn.Linear(512, 384, bias=False)
    lin.weight.data = w.clone().float()
    t = te_linear.TELinear([lin], "mxfp8").to(gpu).train()
    xg = x.to(gpu).requires_grad_(True)
    y = t(xg)
    y.backward(dy.to(gpu))
    torch.cuda.synchronize()
    pad = (rows + 31) // 32 * 32 - rows
    ry, rdx, rdw = orc.linear_fwd_bwd_mx(torch.nn.functional.pad(x, (0, 0, 0, pad)), w,
                                         torch.nn.functional.pad(dy, (0, 0, 0, pad)))
    _close(y, ry[:rows], "mx telinear y")
    _close(xg.grad, rdx[:rows], "mx telinear dx")
    _close(t.weight.grad, rdw, "mx telinear dw")
    t(xg)
    assert t.counts == {"weight_quantizations": 1, "cached_weights": 1}


def _temlp_mx_step(gpu, mlp, x, dy, split, monkeypatch):
    monkeypatch.setenv("BONGARD_TE_SPLIT_GATE_UP", "1" if split else "0")
    t = te_linear.TEMLP(mlp, "mxfp8").to(gpu).train()
    assert t.fused_gate_up != split
    xg = x.to(gpu).requires_grad_(True)
    y = t(xg)
    y.backward(dy.to(gpu))
    torch.cuda.synchronize()
    dwgu = (t.gate_up.weight.grad if not split
            else torch.cat([t.gate_proj.weight.grad, t.up_proj.weight.grad]))
    return y, xg.grad, dwgu, t.down.weight.grad


def test_temlp_mxfp8_fwd_bwd(gpu, monkeypatch):
    """TEMLP under 'mxfp8' against the oracle chain (statistical bar: H and dGU are
    requantized in blocks; where GPU and oracle round a block's largest element to
    neighbouring bf16s across a power of two, the whole block's E8M0 scale moves and its 32
    values requantize on a grid twice as coarse or fine, so single outputs can move by up to
    ~0.1 RMS). The split gate/up layout (BONGARD_TE_SPLIT_GATE_UP=1) quantizes the same
    blocks, so it must reproduce the fused layout bit for bit."""
    hidden, inter, rows = 256, 512, 512
    g = torch.Generator().manual_seed(61)
    mlp = _mlp(hidden, inter, 61)
    wg, wu, wd = (m.weight.detach().clone() for m in (mlp.gate_proj, mlp.up_proj, mlp.down_proj))
    x = torch.randn(rows, hidden, generator=g).to(torch.bfloat16)
    dy = (torch.randn(rows, hidden, generator=g) * 1e-3).to(torch.bfloat16)
    fused = _temlp_mx_step(gpu, mlp, x, dy, False, monkeypatch)
    split = _temlp_mx_step(gpu, mlp, x, dy, True, monkeypatch)
    for a, b in zip(fused, split):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
    ref = orc.mlp_fwd_bwd_mx(x, wg, wu, wd, dy)
    y, dx, dwgu, dwd = fused
    _close_requant(y, ref["y"], "mx temlp y", max_tol=0.10)
    _close_requant(dx, ref["dx"], "mx temlp dx", max_tol=0.2)
    _close_requant(dwgu, ref["dwgu"], "mx temlp dWgu", max_tol=0.2)
    _close_requant(dwd, ref["dwd"], "mx temlp dWd", max_tol=0.2)


def test_fused_mlp_mxfp8_fwd_bwd(gpu):
    hidden, inter, rows = 256, 512, 480
    g = torch.Generator().manual_seed(62)
    mlp = _mlp(hidden, inter, 62)
    norm = T5Gemma2RMSNorm(hidden, eps=1e-6).to(torch.bfloat16)
    with torch.no_grad():
        norm.weight.normal_(std=0.1)
    wg, wu, wd = (m.weight.detach().clone() for m in (mlp.gate_proj, mlp.up_proj, mlp.down_proj))
    nw = norm.weight.detach().clone()
    x = torch.randn(rows, hidden, generator=g).to(torch.bfloat16)
    dy = (torch.randn(rows, hidden, generator=g) * 1e-3).to(torch.bfloat16)
    f = fused_mlp.FusedMLP(mlp, norm, "mxfp8").to(gpu).train()
    xg = x.to(gpu).requires_grad_(True)
    y = f(xg)
    y.backward(dy.to(gpu))
    torch.cuda.synchronize()
    xr = x.clone().requires_grad_(True)
    normed = orc.rmsnorm(xr, nw, 1e-6)
    ref = orc.mlp_fwd_bwd_mx(normed.detach(), wg, wu, wd, dy)
    normed.backward(ref["dx"].to(torch.bfloat16))
    _close_requant(y, ref["y"], "mx fused y", max_tol=0.10)
    _close_requant(xg.grad, xr.grad, "mx fused dx", max_tol=0.2)
    _close_requant(f.fc1_weight.grad, ref["dwgu"], "mx fused dWgu", max_tol=0.2)
    _close_requant(f.fc2_weight.grad, ref["dwd"], "mx fused dWd", max_tol=0.2)
    assert f.state_dict()["_extra_state"].numel() == 0


@pytest.mark.parametrize("tile", ["256x256", "256x160", "160x256", "128x128", "192x256",
                                  "128x64", "64x128", "256x128", "256x256w8", "128x128o2"])
@pytest.mark.parametrize("M,N,K", [(300, 392, 544), (100, 264, 96), (520, 264, 256), (257, 520, 352)])
def test_gemm_mx_every_tile(gpu, monkeypatch, tile, M, N, K):
    """Every block tile's MX variant (those whose stages would overflow the LDS with the
    scale dwords run with one stage fewer), forced through the tuning override: partial tiles in M
    and N, K of one, two, three and five steps with whole and partial last steps, bf16 and fp32
    out, scale rows and planes."""
    monkeypatch.setenv("BONGARD_FP8_GEMM_TILE", tile)
    _mx_gemm_case(gpu, M, N, K, seed=17 + K, bias=K == 352)


def test_gemm_mx_eight_wave_split_k(gpu, monkeypatch):
    """Three K pieces (7, 7 and 6 steps, the last with a partial one) of the eight-wave tile."""
    monkeypatch.setenv("BONGARD_FP8_GEMM_TILE", "256x256w8:3")
    M, N, K = 300, 520, 2528
    assert ops._lib.lib().bf8_gemm_mx_workspace(M, N, K) == 3 * M * N * 4
    _mx_gemm_case(gpu, M, N, K, seed=23, bias=True)


@pytest.mark.parametrize("tile", ["128x128", "256x256w8"])
def test_gemm_mx_inf_and_nan(gpu, monkeypatch, tile):
    """NaN bytes, NaN scales and scales of 2^127 stay in their own row and column of the output,
    and every other element is the oracle's."""
    monkeypatch.setenv("BONGARD_FP8_GEMM_TILE", tile)
    M, N, K = 300, 264, 416
    g = torch.Generator().manual_seed(31)
    qa = ops.quantize_mx(torch.randn(M, K, generator=g).to(torch.bfloat16).to(gpu))
    qb = ops.quantize_mx(torch.randn(N, K, generator=g).to(torch.bfloat16).to(gpu))
    qa.data.view(torch.uint8)[9, K - 1] = 0x7F      # an e4m3 NaN in the partial last step
    qa.scales[258, 1] = 0xFF                        # an E8M0 NaN block
    qb.scales[261, 0] = 254                         # 2^127 against 2^127
    qa.scales[5, 0] = 254
    planes = [_planes_of(q.scales) for q in (qa, qb)]
    y = ops.gemm_mx(qa.data, qa.scales, qb.data, qb.scales)
    yp = ops.gemm_mx(qa.data, None, qb.data, None, a_planes=planes[0], b_planes=planes[1])
    torch.cuda.synchronize()
    y, yp = y.float().cpu(), yp.float().cpu()
    assert torch.equal(y.isnan(), yp.isnan()) and torch.equal(y.nan_to_num(), yp.nan_to_num())
    assert y[[9, 258]].isnan().all() and not y[5, 261].isfinite()
    keep_m, keep_n = torch.ones(M, dtype=torch.bool), torch.ones(N, dtype=torch.bool)
    keep_m[[5, 9, 258]] = False
    keep_n[261] = False
    a8, ae = qa.data.view(torch.uint8).cpu()[keep_m], qa.scales.cpu()[keep_m][:, :K // 32].int()
    b8, be = qb.data.view(torch.uint8).cpu()[keep_n], qb.scales.cpu()[keep_n][:, :K // 32].int()
    ref = orc.scaled_mm_mx(a8, ae, b8, be)
    got = y[keep_m][:, keep_n]
    assert got.isfinite().all()
    excess = ((got - ref).abs() - 0.5 * orc.bf16_ulp(ref)).max().item()
    assert excess <= 0.01 * _rms(ref)


def test_quantize_mx_many_equals_quantize_mx(gpu, monkeypatch):
    """Rowwise MX quantization of several tensors in one launch gives each tensor's own
    bytes and scales (formats mixed, a ragged row count, an empty tensor skipped); the MX
    gated MLP's inference forward, which uses it, equals its training forward bit for bit."""
    from bongard_amd import linear
    g = torch.Generator().manual_seed(3)
    xs = [torch.randn(300, 2560, generator=g).to(torch.bfloat16).to(gpu),
          (torch.randn(8192, 4096, generator=g) * 40).to(torch.bfloat16).to(gpu),
          torch.randn(64, 96, generator=g).to(torch.bfloat16).to(gpu),
          torch.empty(0, 64, dtype=torch.bfloat16, device=gpu)]
    xs[2][3, 5] = float("nan")
    fmts = [ops.E4M3, ops.E5M2, ops.E4M3, ops.E4M3]
    qs = ops.quantize_mx_many(xs, fmts)
    for x, q, f in zip(xs[:3], qs, fmts):
        r = ops.quantize_mx(x, f)
        assert torch.equal(q.data.view(torch.uint8), r.data.view(torch.uint8))
        assert torch.equal(q.scales, r.scales)
    assert qs[3].data.numel() == 0
    with pytest.raises(RuntimeError):
        ops.quantize_mx_many([xs[0], torch.zeros(32, 48, dtype=torch.bfloat16, device=gpu)])
    # the inference forwards (no_grad) of the MX MLP and linear on trainable weights take
    # the shared launch; their outputs equal the training forwards' bit for bit
    calls = []
    real = ops.quantize_mx_many

    def counted(*a, **k):
        calls.append(1)
        return real(*a, **k)

    monkeypatch.setattr(ops, "quantize_mx_many", counted)
    x = torch.randn(256, 256, generator=g).to(torch.bfloat16).to(gpu)
    w_gu = torch.nn.Parameter((torch.randn(1024, 256, generator=g) * 0.02).to(torch.bfloat16).to(gpu))
    w_d = torch.nn.Parameter((torch.randn(256, 512, generator=g) * 0.014).to(torch.bfloat16).to(gpu))
    y_train = linear.Fp8GegluMlpMxFunction.apply(x, w_gu, w_d, None, None, 512)
    assert len(calls) == 0
    with torch.no_grad():
        y_inf = linear.Fp8GegluMlpMxFunction.apply(x, w_gu, w_d, None, None, 512)
    assert len(calls) == 1
    assert torch.equal(y_train.detach(), y_inf)
    w_o = torch.nn.Parameter(w_d.detach().t().contiguous())
    y_train = linear.Fp8LinearMxFunction.apply(x, w_o, None)
    with torch.no_grad():
        y_inf = linear.Fp8LinearMxFunction.apply(x, w_o, None)
    assert len(calls) == 2
    assert torch.equal(y_train.detach(), y_inf)


def test_module_weight_keeps_scale_rows(gpu):
    """The cached MXFP8 weight a module hands out still holds its scales as rows, for a caller's
    own ``gemm_mx`` on them."""
    g = torch.Generator().manual_seed(5)
    lin = torch.nn.Linear(160, 96, bias=False, dtype=torch.bfloat16)
    with torch.no_grad():
        lin.weight.copy_(torch.randn(96, 160, generator=g) * 0.02)
    layer = te_linear.TELinear([lin], "mxfp8").to(gpu)
    q = layer.fp8_weight(True)
    r = ops.quantize_mx(layer.weight.detach(), rowwise=True, colwise=True)
    for name in ("data", "scales", "data_t", "scales_t", "planes", "planes_t"):
        assert torch.equal(getattr(q, name).view(torch.uint8), getattr(r, name).view(torch.uint8))
    x = ops.quantize_mx(torch.randn(33, 160, generator=g).to(torch.bfloat16).to(gpu))
    assert torch.equal(ops.gemm_mx(x.data, x.scales, q.data, q.scales),
                       ops.gemm_mx(x.data, None, q.data, None, a_planes=x.planes,
                                   b_planes=q.planes))


@pytest.mark.parametrize("hidden,inter", [(256, 384), (160, 128)])
def test_weights_of_scale_rows_alone(gpu, hidden, inter):
    """MXFP8 weights put together from scale rows, without planes (as from the C quantizer's
    outputs; here with rows wider than the scales), run the linear and the gated MLP with the
    outputs and gradients of a weight that holds both, bit for bit."""
    from bongard_amd import linear
    g = torch.Generator().manual_seed(hidden)
    M = 96
    x = torch.randn(M, hidden, generator=g).to(torch.bfloat16).to(gpu)
    w_gu = (torch.randn(2 * inter, hidden, generator=g) * 0.02).to(torch.bfloat16).to(gpu)
    w_d = (torch.randn(hidden, inter, generator=g) * 0.02).to(torch.bfloat16).to(gpu)
    dy = (torch.randn(M, hidden, generator=g) * 1e-3).to(torch.bfloat16).to(gpu)

    def rows_alone(q):
        def wide(s):
            w = torch.full((s.shape[0], s.shape[1] + 8), 0xFF, dtype=torch.uint8, device=gpu)
            w[:, :s.shape[1]] = s
            return w[:, :s.shape[1]]
        return ops.MxFp8Tensor(q.data, wide(q.scales), q.data_t, wide(q.scales_t), q.fmt, q.rows,
                               q.cols)

    def both(q):
        return q

    out = []
    for form in (both, rows_alone):
        gu_q, d_q = form(linear.quantize_weight_mx(w_gu)), form(linear.quantize_weight_mx(w_d))
        xg, gu, wd = (t.detach().clone().requires_grad_(True) for t in (x, w_gu, w_d))
        y = linear.Fp8GegluMlpMxFunction.apply(xg, gu, wd, gu_q, d_q, inter)
        res = [y, *torch.autograd.grad(y, [xg, gu, wd], dy)]
        h = torch.randn(M, inter, generator=torch.Generator().manual_seed(3)).to(torch.bfloat16)
        hg = h.to(gpu).requires_grad_(True)
        z = linear.Fp8LinearMxFunction.apply(hg, wd, d_q)
        res += [z, *torch.autograd.grad(z, [hg, wd], dy)]
        with torch.no_grad():
            res.append(linear.Fp8LinearMxFunction.apply(hg, wd, d_q))
        out.append(res)
    torch.cuda.synchronize()
    for a, b in zip(*out):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
