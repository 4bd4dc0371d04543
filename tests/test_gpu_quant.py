"""GPU parity of amax / scale / cast (+ transposed copy) against the CPU oracle.

The bar is bit-exact: every fp8 byte, amax, scale and scale_inv must equal the oracle's.
"""

import numpy as np
import pytest
import torch

from bongard_amd import _lib, ops, workloads
from oracle import fp8_oracle as orc

pytestmark = pytest.mark.gpu


def _bytes(t):
    return t.view(torch.uint8).cpu()


def _check_quant(x_cpu, fmt, dev, transpose=True):
    q = ops.quantize(x_cpu.to(dev), fmt, rowwise=True, transpose=transpose)
    torch.cuda.synchronize()
    ref_q, ref_a, ref_s, ref_si = orc.quantize(x_cpu.reshape(-1, x_cpu.shape[-1]), fmt)
    meta = q.meta.cpu()
    assert meta[0].view(torch.int32) == ref_a.view(torch.int32), (meta[0], ref_a)
    assert meta[1].view(torch.int32) == ref_s.view(torch.int32), (meta[1], ref_s)
    assert meta[2].view(torch.int32) == ref_si.view(torch.int32), (meta[2], ref_si)
    got = _bytes(q.data)
    mism = (got != ref_q).sum().item()
    assert mism == 0, f"{mism} fp8 bytes differ"
    if transpose:
        assert torch.equal(_bytes(q.data_t), ref_q.t().contiguous())
    return q


@pytest.mark.parametrize("fmt", [ops.E4M3, ops.E5M2])
def test_config1_quantize_bit_exact(gpu, fmt):
    c = workloads.config1()
    _check_quant(c["x"], fmt, gpu)
    _check_quant(c["w"], fmt, gpu)


@pytest.mark.parametrize("fmt", [ops.E4M3, ops.E5M2])
@pytest.mark.parametrize("scale", [1.0, 6.9457, 0.0001220703125, 3.0e4, 4.48e14])
def test_every_bf16_pattern(gpu, fmt, scale):
    """All 65,536 bf16 bit patterns (NaN, inf, subnormals, both zeros) at a fixed scale."""
    bits = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    x = bits.reshape(256, 256)
    meta = torch.tensor([0.0, scale, 1.0 / scale, 0.0], dtype=torch.float32)
    q = ops.cast(x.to(gpu), meta.to(gpu), fmt, rowwise=True, transpose=True)
    torch.cuda.synchronize()
    ref = orc.cast(x, meta[1], fmt)
    got = _bytes(q.data)
    bad = (got != ref).nonzero()
    assert bad.numel() == 0, f"{bad.shape[0]} mismatches, first at {bad[:4].tolist()}: " \
        f"x={x[tuple(bad[0].tolist())]} got={got[tuple(bad[0].tolist())]} ref={ref[tuple(bad[0].tolist())]}"
    assert torch.equal(_bytes(q.data_t), ref.t().contiguous())


@pytest.mark.parametrize("shape", [(1, 16), (3, 48), (31, 2560), (100, 272), (513, 2560),
                                   (64, 64), (65, 80), (2048, 16)])
def test_ragged_shapes(gpu, shape):
    g = torch.Generator().manual_seed(sum(shape))
    x = (torch.randn(*shape, generator=g) * 3).to(torch.bfloat16)
    _check_quant(x, ops.E4M3, gpu)
    _check_quant(x, ops.E5M2, gpu)


@pytest.mark.parametrize("shape", [(8256, 4160), (8261, 4160)])
def test_transpose_grid_wraps_with_odd_tile_counts(gpu, shape):
    # more 64 x 64 tiles than one pass of the transposing grid (4,096 waves), an odd number
    # of tile columns, and an odd tile-row count (8256 rows: 129 tile rows; 8261: a ragged
    # last tile row and out_t rows that are not 16-byte aligned): the tile-row-pair walk
    # must still cover every tile once
    g = torch.Generator().manual_seed(shape[0])
    x = (torch.randn(*shape, generator=g) * 2).to(torch.bfloat16)
    _check_quant(x, ops.E4M3, gpu)


def test_odd_total_rowwise_only(gpu):
    # n % 16 != 0 exercises the scalar tail of the row-major cast (no transpose).
    g = torch.Generator().manual_seed(7)
    x = torch.randn(3, 7, generator=g).to(torch.bfloat16)
    _check_quant(x, ops.E4M3, gpu, transpose=False)


def test_special_values(gpu):
    x = torch.zeros(64, 64, dtype=torch.bfloat16)
    _check_quant(x, ops.E4M3, gpu)  # amax 0 -> scale 448 / 1e-12
    x[3, 5] = float("inf")
    _check_quant(x, ops.E4M3, gpu)  # amax inf -> scale 0, inf * 0 -> NaN byte
    y = torch.randn(64, 64).to(torch.bfloat16)
    y[7, 9] = float("nan")
    _check_quant(y, ops.E4M3, gpu)  # NaN amax -> NaN scale
    _check_quant(y, ops.E5M2, gpu)


def test_large_amax_partials(gpu):
    # more elements than one pass of the amax grid: exercises the grid-stride loop
    g = torch.Generator().manual_seed(11)
    x = torch.randn(4096, 2560, generator=g).to(torch.bfloat16)
    x[4000, 2500] = -77.5
    _check_quant(x, ops.E4M3, gpu)


def test_delayed_scaling_matches_closed_form(gpu):
    L = 16
    st = ops.new_delayed_state(L, gpu)
    ref = orc.DelayedScaling(L, ops.E4M3)
    g = torch.Generator().manual_seed(5)
    for step in range(40):
        x = (torch.randn(128, 256, generator=g) * (1 + (step % 7))).to(torch.bfloat16)
        meta = ops.delayed_scale_begin(st, L, ops.E4M3)
        q = ops.cast(x.to(gpu), meta, ops.E4M3)
        parts = ops.amax(x.to(gpu))
        ops.delayed_scale_end(st, L, parts)
        s, si = ref.begin()
        ref_q = orc.cast(x, torch.tensor(s), ops.E4M3)
        ref.end(float(orc.amax(x)))
        torch.cuda.synchronize()
        m = meta.cpu()
        assert m[1].item() == float(s) and m[2].item() == float(si), (step, m, s, si)
        assert torch.equal(_bytes(q.data), ref_q), step
    assert np.array_equal(st[:L].cpu().numpy(), ref.history)


def test_quantize_many_equals_quantize(gpu):
    """Several tensors quantized in two shared launches give each tensor's own bytes and
    meta: against the oracle for the small ones, against the single-tensor quantization
    (itself pinned to the oracle above) for one large enough to hit the partials cap;
    formats mixed, a ragged size, an empty tensor (its meta left untouched)."""
    g = torch.Generator().manual_seed(11)
    small = [torch.randn(512, 2560, generator=g).to(torch.bfloat16),
             (torch.randn(1, 1007, generator=g) * 300).to(torch.bfloat16),
             torch.randn(256, 4096, generator=g).to(torch.bfloat16)]
    small[2][7, 9] = float("inf")
    big = torch.randn(8192, 4608, generator=g).to(torch.bfloat16).to(gpu)
    empty = torch.empty(0, 2560, dtype=torch.bfloat16, device=gpu)
    fmts = [ops.E4M3, ops.E5M2, ops.E4M3, ops.E5M2, ops.E4M3]
    sentinel = torch.full((4,), -7.0, device=gpu)
    metas = [ops.new_meta(gpu) for _ in range(3)] + [ops.new_meta(gpu), sentinel.clone()]
    xs = [t.to(gpu) for t in small] + [big, empty]
    qs = ops.quantize_many(xs, fmts, metas=metas)
    torch.cuda.synchronize()
    for t, q, f in zip(small, qs[:3], fmts[:3]):
        ref_q, ref_a, ref_s, ref_si = orc.quantize(t, f)
        meta = q.meta.cpu()
        assert meta[0].view(torch.int32) == ref_a.view(torch.int32)
        assert meta[1].view(torch.int32) == ref_s.view(torch.int32)
        assert meta[2].view(torch.int32) == ref_si.view(torch.int32)
        assert torch.equal(_bytes(q.data), ref_q)
    one = ops.quantize(big, ops.E5M2)
    assert torch.equal(qs[3].data.view(torch.uint8), one.data.view(torch.uint8))
    assert torch.equal(qs[3].meta, one.meta)
    assert torch.equal(qs[4].meta, sentinel)
    # power-of-two scales, one format for all
    qp = ops.quantize_many(xs[:2], ops.E4M3, pow2=True)
    for x, q in zip(xs[:2], qp):
        r = ops.quantize(x, ops.E4M3, pow2=True)
        assert torch.equal(q.data.view(torch.uint8), r.data.view(torch.uint8))
        assert torch.equal(q.meta, r.meta)


@pytest.mark.parametrize("rows,cols", [(1, 1), (3, 5), (1, 16), (7, 33), (64, 256), (65, 2560),
                                       (1, 16385), (64, 1024), (4096, 16), (1, 64 * 1024 + 1),
                                       (192, 1024), (193, 1024)])
@pytest.mark.parametrize("special", [None, "inf", "nan", "zero"])
def test_quantize_one_launch_equals_two(gpu, rows, cols, special):
    """A small tensor's one-launch quantization (up to 192 x 1024 elements) and the first size past
    it against the amax and cast passes of quantize_many: the same bytes and meta."""
    x = torch.randn(rows, cols, generator=torch.Generator().manual_seed(rows + cols)).bfloat16()
    if special == "zero":
        x.zero_()
    elif special:
        x.view(-1)[-1] = float(special)   # the last element: the tail of n % 16
    x = x.to(gpu)
    for fmt in (ops.E4M3, ops.E5M2):
        for pow2 in (False, True):
            one = ops.quantize(x, fmt, pow2=pow2)
            two = ops.quantize_many([x], fmt, pow2=pow2)[0]
            torch.cuda.synchronize()
            assert torch.equal(one.data.view(torch.uint8), two.data.view(torch.uint8))
            assert torch.equal(one.meta.view(torch.int32), two.meta.view(torch.int32))


@pytest.mark.parametrize("n", [1, 16, 16385, 64 * 1024, 64 * 1024 + 16, 192 * 1024, 192 * 1024 + 8])
def test_quantize_leaves_the_amax_partials(gpu, n):
    """bf8_quantize_bf16 leaves the tensor's amax in the partials it was given, in one launch or
    two: a second cast of x from them equals its own quantization, and no slot past
    bf8_amax_partials is written."""
    L = _lib.lib()
    x = torch.randn(1, n, generator=torch.Generator().manual_seed(n)).bfloat16().to(gpu)
    np_ = L.bf8_amax_partials(n)
    parts = torch.full((np_ + 4,), 0x7F123456, dtype=torch.int32, device=gpu)
    out, meta = torch.empty(n, dtype=torch.uint8, device=gpu), ops.new_meta(gpu)
    _lib.check(L.bf8_quantize_bf16(x.data_ptr(), 1, n, ops.E4M3, out.data_ptr(), None,
                                   meta.data_ptr(), parts.data_ptr(),
                                   torch.cuda.current_stream().cuda_stream), "bf8_quantize_bf16")
    torch.cuda.synchronize()
    assert (parts[np_:] == 0x7F123456).all()
    assert parts[:np_].max().item() == meta[0].view(torch.int32).item()
    second = ops.cast_partials(x, parts[:np_], ops.E5M2)
    want = ops.quantize_many([x], ops.E5M2)[0]
    assert torch.equal(second.data.view(torch.uint8), want.data.view(torch.uint8))
    assert torch.equal(second.meta, want.meta)


@pytest.mark.parametrize("n", [64 * 1024, 64 * 1024 + 16, 164 * 1024, 192 * 1024])
def test_quantize_captured_in_a_graph(gpu, n):
    """Captured in a graph, tensors past 64 x 1024 elements take the two launches, whose device
    time is the shorter (their partials are then the amax pass's, slot for slot); every replay, on
    new values and between eager calls of the one-launch path, gives the eager bytes and meta."""
    L = _lib.lib()
    x = torch.zeros(1, n, dtype=torch.bfloat16, device=gpu)
    parts = torch.zeros(L.bf8_amax_partials(n), dtype=torch.int32, device=gpu)
    out, meta = torch.empty(n, dtype=torch.uint8, device=gpu), ops.new_meta(gpu)

    def call():
        _lib.check(L.bf8_quantize_bf16(x.data_ptr(), 1, n, ops.E4M3, out.data_ptr(), None,
                                       meta.data_ptr(), parts.data_ptr(),
                                       torch.cuda.current_stream().cuda_stream), "quantize")

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        call()
    for seed in range(3):
        x.copy_(torch.randn(1, n, generator=torch.Generator().manual_seed(seed)).bfloat16() * 3 ** seed)
        want = ops.quantize(x)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want.data.view(torch.uint8).view(-1))
        assert torch.equal(meta, want.meta)
        assert torch.equal(parts, ops.amax(x)) == (n > 64 * 1024)


def test_quantize_many_rejects_bad_lists(gpu):
    x = torch.randn(64, 64, device=gpu).to(torch.bfloat16)
    with pytest.raises(ValueError):
        ops.quantize_many([])
    with pytest.raises(ValueError):
        ops.quantize_many([x] * 9)
    with pytest.raises(ValueError):
        ops.quantize_many([x, x], [ops.E4M3])
