"""GPU parity of the dequant-fused GEMV / skinny GEMM kernels against the oracle's evaluator
semantics (dequantize to f32, then eval_matmul_2d): |y - ref| <= 1e-3 + 1e-2 * |ref|, the
north-star tolerance for bf16 accumulation."""
import numpy as np
import pytest
import torch

import oracle_lib as O
from castforge_amd import ops, synth

pytestmark = pytest.mark.gpu

RTOL, ATOL = 1e-2, 1e-3


def _close(y, ref):
    y = y.float().cpu().numpy()
    err = np.abs(y - ref)
    bound = ATOL + RTOL * np.abs(ref)
    bad = err > bound
    assert not bad.any(), f"{bad.sum()} / {bad.size} outside tol; max err {err.max():.3e}"


def _x(seed, m, k, dev):
    xb = synth.activations_bf16(seed, 7, m, k)
    return xb, torch.from_numpy(xb.view(np.int16)).view(torch.bfloat16).to(dev)


@pytest.mark.parametrize("m", [1, 2, 8, 16, 17, 33, 64])
@pytest.mark.parametrize("n,k", [(48, 256), (100, 1024), (64, 11008), (4096, 4096)])
@pytest.mark.parametrize("out", [torch.float32, torch.bfloat16])
def test_w4a16_skinny(cuda, m, n, k, out):
    w = synth.weight(51, 1, n, k)
    codes, scales, zeros = O.quantize_int4g(w, 128)
    xb, x = _x(52, m, k, cuda)
    p = ops.Int4Packed(torch.from_numpy(codes.view(np.int32)).to(cuda),
                       torch.from_numpy(scales.view(np.float16)).to(cuda),
                       torch.from_numpy(zeros.view(np.int32)).to(cuda), n, k, 128)
    y = ops.gemm_w4a16(x, p, out)
    torch.cuda.synchronize()
    _close(y, O.gemm_w4a16(xb, codes, scales, zeros, n, k, 128))


@pytest.mark.parametrize("m,group,k", [(3, 64, 512), (20, 128, 256), (1, 32, 1000), (5, 256, 512)])
def test_w4a16_generic_paths(cuda, m, group, k):
    n = 37
    w = synth.weight(53, 1, n, k)
    xb, x = _x(54, m, k, cuda)
    p = ops.quantize_int4g(torch.from_numpy(w).to(cuda), group)
    y = ops.gemm_w4a16(x, p, torch.float32)
    ref = O.gemm_w4a16(xb, p.codes.cpu().numpy().view(np.uint32), p.scales.cpu().numpy().view(np.uint16),
                       p.zeros.cpu().numpy().view(np.uint32), n, k, group)
    _close(y, ref)


@pytest.mark.parametrize("m", [1, 5, 16, 17, 32, 33])
@pytest.mark.parametrize("gran", ["channel", "tensor"])
@pytest.mark.parametrize("n,k", [(40, 192), (4096, 4096), (33, 11008)])
def test_w8a16(cuda, m, gran, n, k):
    w = synth.weight(61, 1, n, k)
    xb, x = _x(62, m, k, cuda)
    q, s = ops.quantize_int8(torch.from_numpy(w).to(cuda), 8, gran, "half_even")
    y = ops.gemm_w8a16(x, q, s, gran, torch.float32)
    sc = s.cpu().numpy()
    sc = sc if gran == "channel" else np.full(n, sc[0], np.float32)
    _close(y, O.gemm_w8a16(xb, q.cpu().numpy(), sc))


@pytest.mark.parametrize("m", [1, 16, 17, 40, 64])
@pytest.mark.parametrize("block", [64, 32, 16])
def test_nf4(cuda, m, block):
    n, k = 96, 1024
    w = synth.weight(71, 1, n, k)
    xb, x = _x(72, m, k, cuda)
    p = ops.quantize_nf4(torch.from_numpy(w).to(cuda), block)
    y = ops.gemm_nf4(x, p, torch.float32)
    ref = O.gemm_nf4(xb, p.codes.cpu().numpy().view(np.uint32), p.absmax.cpu().numpy(), n, k, block)
    _close(y, ref)


def test_w4a16_batched_block_m1(cuda):
    """The bench's single launch: 7 projections of one LLaMA-7B block at M=1."""
    xs, ps, ys, refs = [], [], [], []
    for tid, (name, n, k) in enumerate(synth.LLAMA7B_BLOCK):
        w = synth.weight(0, tid, n, k)
        codes, scales, zeros = O.quantize_int4g(w, 128)
        xb, x = _x(100 + tid, 1, k, cuda)
        ps.append(ops.Int4Packed(torch.from_numpy(codes.view(np.int32)).to(cuda),
                                 torch.from_numpy(scales.view(np.float16)).to(cuda),
                                 torch.from_numpy(zeros.view(np.int32)).to(cuda), n, k, 128))
        xs.append(x)
        ys.append(torch.empty((1, n), dtype=torch.bfloat16, device=cuda))
        refs.append(O.gemm_w4a16(xb, codes, scales, zeros, n, k, 128))
    ops.gemv_w4a16_batched(xs, ps, ys)
    torch.cuda.synchronize()
    for y, ref in zip(ys, refs):
        _close(y, ref)


def test_empty_and_degenerate(cuda):
    p = ops.quantize_int4g(torch.zeros((0, 256), device=cuda), 128)
    x = torch.zeros((1, 256), dtype=torch.bfloat16, device=cuda)
    assert ops.gemm_w4a16(x, p).shape == (1, 0)
    w = torch.zeros((16, 256), device=cuda)
    p = ops.quantize_int4g(w, 128)
    y = ops.gemm_w4a16(torch.ones((1, 256), dtype=torch.bfloat16, device=cuda), p, torch.float32)
    assert torch.all(y == 0)


@pytest.mark.parametrize("gran", ["channel", "tensor"])
@pytest.mark.parametrize("m", [1, 4])
def test_w8a16_batched(cuda, gran, m):
    """One launch over several INT8 problems: same bits as one call per problem, oracle tolerance."""
    shapes = [(40, 192), (4096, 4096), (33, 11008), (100, 64)]
    xs, qs, ys, singles, refs = [], [], [], [], []
    for i, (n, k) in enumerate(shapes):
        w = synth.weight(400 + i, 1, n, k)
        xb, x = _x(410 + i, m, k, cuda)
        q, s = ops.quantize_int8(torch.from_numpy(w).to(cuda), 8, gran, "half_even")
        xs.append(x)
        qs.append((q, s))
        ys.append(torch.empty((m, n), dtype=torch.float32, device=cuda))
        singles.append(ops.gemm_w8a16(x, q, s, gran, torch.float32))
        sc = s.cpu().numpy()
        refs.append(O.gemm_w8a16(xb, q.cpu().numpy(), sc if gran == "channel" else np.full(n, sc[0], np.float32)))
    ops.gemv_w8a16_batched(xs, qs, ys, gran)
    for y, y1, ref in zip(ys, singles, refs):
        assert torch.equal(y, y1)
        _close(y, ref)


@pytest.mark.parametrize("block", [64, 32])
def test_nf4_batched(cuda, block):
    shapes = [(96, 1024), (11008, 4096), (4096, 11008), (7, 512)]
    xs, ps, ys, singles, refs = [], [], [], [], []
    for i, (n, k) in enumerate(shapes):
        w = synth.weight(420 + i, 1, n, k)
        xb, x = _x(430 + i, 1, k, cuda)
        p = ops.quantize_nf4(torch.from_numpy(w).to(cuda), block)
        xs.append(x)
        ps.append(p)
        ys.append(torch.empty((1, n), dtype=torch.float32, device=cuda))
        singles.append(ops.gemm_nf4(x, p, torch.float32))
        refs.append(O.gemm_nf4(xb, p.codes.cpu().numpy().view(np.uint32), p.absmax.cpu().numpy(), n, k, block))
    ops.gemv_nf4_batched(xs, ps, ys)
    for y, y1, ref in zip(ys, singles, refs):
        assert torch.equal(y, y1)
        _close(y, ref)


@pytest.mark.parametrize("fmt", ["int4", "int8", "nf4"])
@pytest.mark.parametrize("m", [17, 40, 64])
def test_batched_mid_m(cuda, fmt, m):
    """M = 17..64 in one batched launch of the K-split kernel: within tolerance of the oracle, and equal to
    one call per problem."""
    shapes = [(96, 1024), (300, 2048), (64, 4096), (7, 512)]
    xs, ps, ys, refs = [], [], [], []
    for i, (n, k) in enumerate(shapes):
        w = torch.from_numpy(synth.weight(700 + i, 1, n, k)).to(cuda)
        xb, x = _x(710 + i, m, k, cuda)
        xs.append(x)
        ys.append(torch.empty((m, n), dtype=torch.float32, device=cuda))
        if fmt == "int4":
            p = ops.quantize_int4g(w, 128)
            refs.append(O.gemm_w4a16(xb, p.codes.cpu().numpy().view(np.uint32), p.scales.cpu().numpy().view(np.uint16),
                                     p.zeros.cpu().numpy().view(np.uint32), n, k, 128))
        elif fmt == "int8":
            p = ops.quantize_int8(w, 8, "channel", "half_even")
            refs.append(O.gemm_w8a16(xb, p[0].cpu().numpy(), p[1].cpu().numpy()))
        else:
            p = ops.quantize_nf4(w, 64)
            refs.append(O.gemm_nf4(xb, p.codes.cpu().numpy().view(np.uint32), p.absmax.cpu().numpy(), n, k, 64))
        ps.append(p)
    if fmt == "int4":
        ops.gemv_w4a16_batched(xs, ps, ys)
        singles = [ops.gemm_w4a16(x, p, torch.float32) for x, p in zip(xs, ps)]
    elif fmt == "int8":
        ops.gemv_w8a16_batched(xs, ps, ys, "channel")
        singles = [ops.gemm_w8a16(x, q, s, "channel", torch.float32) for x, (q, s) in zip(xs, ps)]
    else:
        ops.gemv_nf4_batched(xs, ps, ys)
        singles = [ops.gemm_nf4(x, p, torch.float32) for x, p in zip(xs, ps)]
    for y, y1, ref in zip(ys, singles, refs):
        assert torch.equal(y, y1)
        _close(y, ref)
        _close(y1, ref)


def _nf4_on(dev, seed, n, k):
    """NF4 weight drawn on the device: packed, and dequantized in float64."""
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    p = ops.quantize_nf4(torch.randn((n, k), generator=g, device=dev) * 0.02, 64)
    return p, ops.dequantize_nf4(p).double()


@pytest.mark.parametrize("m", [17, 32, 40, 64])
@pytest.mark.parametrize("k", [256, 384, 512, 640, 768, 1152, 1408, 6208, 6400, 6464])
def test_nf4_partial_step_groups(cuda, k, m):
    """nf4_mfma_kernel (M = 17..64 with more than one 64 x 64 tile per CU) with every remainder of the K loop's
    groups of six 64-wide steps per K part: 2..11 steps in two parts, 25 and 26 in four of equal and unequal
    length (K > 6144), on weights no earlier call has brought into the caches; in a batch with a smaller
    problem, which qsplit_kernel takes.  Both are against float64 and give the bits of their single calls."""
    n = 64 * torch.cuda.get_device_properties(cuda).multi_processor_count + 70
    (p, wd), (q, qd) = _nf4_on(cuda, 740 + k, n, k), _nf4_on(cuda, 741 + k, 97, k)
    _, x = _x(750 + k, m, k, cuda)
    torch.empty(1 << 28, dtype=torch.uint8, device=cuda).zero_()  # 256 MB through the caches
    y = ops.gemm_nf4(x, p, torch.float32)
    ys = [torch.empty((m, n), device=cuda), torch.empty((m, 97), device=cuda)]
    ops.gemv_nf4_batched([x, x], [p, q], ys)
    assert torch.equal(ys[0], y)
    assert torch.equal(ys[1], ops.gemm_nf4(x, q, torch.float32))
    x64 = x.double()
    for got, w in ((ys[0], wd), (ys[1], qd)):
        # T_hi + T_lo is within 2^-17 of T, the dequantized weight within 2^-24; f32 sums: one rounding an
        # MFMA step of 16, a scale every 64, the K parts or waves
        bound = (2.0 ** -17 + (k / 8 + k / 64 + 10) * 2.0 ** -24) * (x64.abs() @ w.abs().t())
        assert bool(((got.double() - x64 @ w.t()).abs() <= bound).all())


@pytest.mark.parametrize("m", [2, 3, 16, 17, 33, 48, 64])
@pytest.mark.parametrize("gran", ["channel", "tensor"])
def test_w8a16_skinny(cuda, monkeypatch, m, gran):
    """The INT8 skinny kernel at each of its tile counts, with row remainders: at K = 2^23, beyond the
    K-split kernel's 32-bit offsets, and (M > 16) with that kernel turned off.  Activations of one in 2048 and
    a power-of-two scale make every sum of the long rows an integer below 2^24: exact."""
    for n, k in [(35, 1 << 23)] if m <= 16 else [(35, 1 << 23), (300, 1088)]:
        monkeypatch.delenv("CASTFORGE_PREFILL_I4", raising=False)
        if k < 1 << 23:
            monkeypatch.setenv("CASTFORGE_PREFILL_I4", "0")
        g = torch.Generator(device=cuda)
        g.manual_seed(760 + m)
        q = torch.randint(-127, 128, (n, k), generator=g, device=cuda, dtype=torch.int8)
        s = torch.full((n if gran == "channel" else 1,), 0.5, device=cuda)
        if k < 1 << 23:
            _, x = _x(761, m, k, cuda)
        else:
            x = torch.zeros((m, k), dtype=torch.bfloat16, device=cuda)
            x[:, 1023::2048] = torch.randint(-4, 5, (m, k // 2048), generator=g, device=cuda).to(torch.bfloat16)
        y = torch.empty((m, n), device=cuda)
        ops.gemv_w8a16_batched([x], [(q, s)], [y], gran)
        cols = x.abs().amax(0) > 0
        x64, w64 = x[:, cols].double(), q[:, cols].double() * 0.5
        ref, mag = x64 @ w64.t(), x64.abs() @ w64.abs().t()
        if k < 1 << 23:  # two f16 pieces of x a chunk: one rounding an MFMA step and piece, a scale every 64
            assert bool(((y.double() - ref).abs() <= (k / 8 + k / 64 + 10) * 2.0 ** -24 * mag).all())
        else:
            assert float(mag.max()) < 2 ** 23 and torch.equal(y.double(), ref)


def test_nf4_batched_rejects_mixed_blocks(cuda):
    ps = [ops.quantize_nf4(torch.zeros((16, 256), device=cuda), b) for b in (64, 32)]
    xs = [torch.zeros((1, 256), dtype=torch.bfloat16, device=cuda)] * 2
    ys = [torch.empty((1, 16), dtype=torch.float32, device=cuda) for _ in ps]
    with pytest.raises(Exception, match="block size"):
        ops.gemv_nf4_batched(xs, ps, ys)


def test_batched_wrappers_reject_mixed_or_strided_outputs(cuda):
    """Every batched wrapper validates each y (one dtype for the batch, contiguous, [M, n], on
    x's device) before the launch: the C ABI takes a single y_dtype, so a bf16 y after an f32
    one would be written 4 bytes per element."""
    n, k = 32, 256
    w = torch.from_numpy(synth.weight(5, 1, n, k)).to(cuda)
    x = torch.zeros((1, k), dtype=torch.bfloat16, device=cuda)
    p4 = ops.quantize_int4g(w, 128)
    q8 = ops.quantize_int8(w, 8, "channel", "half_even")
    nf = ops.quantize_nf4(w, 64)
    f32y = lambda: torch.empty((1, n), dtype=torch.float32, device=cuda)  # noqa: E731
    bad_sets = [
        ([f32y(), torch.empty((1, n), dtype=torch.bfloat16, device=cuda)], "one dtype"),
        ([f32y(), torch.empty((1, 2 * n), dtype=torch.float32, device=cuda)[:, ::2]], "contiguous"),
        ([f32y(), torch.empty((1, n + 1), dtype=torch.float32, device=cuda)], r"\[M, n\]"),
    ]
    calls = [
        lambda ys: ops.gemv_w4a16_batched([x, x], [p4, p4], ys),
        lambda ys: ops.gemv_w8a16_batched([x, x], [q8, q8], ys, "channel"),
        lambda ys: ops.gemv_nf4_batched([x, x], [nf, nf], ys),
    ]
    for call in calls:
        for ys, msg in bad_sets:
            with pytest.raises(ValueError, match=msg):
                call(ys)
        ys = [f32y(), f32y()]
        call(ys)  # a valid batch still runs
    torch.cuda.synchronize()
