"""GPU parity of the K-split MFMA kernel (M >= 2, small and mid-sized) against float64 products of
the dequantized weights, at sizes that reach each of its tiles and their remainders."""
import numpy as np
import pytest
import torch

from castforge_amd import ffi, ops, synth

pytestmark = pytest.mark.gpu

# (m, n): 32 x 32 tiles (M <= 32; few tiles); 32 (n) x 64 (M <= 64, M > 64); 64 x 64 (M <= 64,
# M > 64); 64 (n) x 128; one row and column past or short of a tile
SHAPES = [(2, 1), (31, 65), (19, 9000), (33, 64), (64, 97), (40, 4200), (70, 2803), (40, 9000), (130, 4000), (300, 3301)]


def _weight(fmt, n, k, cuda):
    wd, run, run_batch, p = _packed(fmt, n, k, cuda)
    return wd, run, lambda x, y: run_batch([x], [p], [y])


def _packed(fmt, n, k, cuda):
    """Dequantized weight, single call (x, out dtype), batched call (xs, packed, ys), packed weight."""
    w = torch.from_numpy(synth.weight(31, n, n, k)).to(cuda)
    if fmt.startswith("int4"):
        p = ops.quantize_int4g(w, int(fmt[5:]))
        return ops.dequantize_int4g(p), lambda x, o: ops.gemm_w4a16(x, p, o), ops.gemv_w4a16_batched, p
    if fmt.startswith("int8"):
        gran = fmt[5:]
        q, s = ops.quantize_int8(w, 8, gran)
        return (ops.dequantize_int8(q, s, gran), lambda x, o: ops.gemm_w8a16(x, q, s, gran, o),
                lambda xs, ps, ys: ops.gemv_w8a16_batched(xs, ps, ys, gran), (q, s))
    if fmt.startswith("nf4"):
        p = ops.quantize_nf4(w, int(fmt[4:]))
        return ops.dequantize_nf4(p), lambda x, o: ops.gemm_nf4(x, p, o), ops.gemv_nf4_batched, p
    ty, size = (ffi.GGML_Q4_0, 18) if fmt == "q4_0" else (ffi.GGML_Q8_0, 34)
    rng = np.random.default_rng(n + k)
    raw = rng.integers(0, 256, (n * k // 32, size), dtype=np.uint8)
    raw[:, :2] = rng.uniform(1e-3, 2e-3, (n * k // 32, 1)).astype(np.float16).view(np.uint8)
    p = ops.gguf_repack(ty, torch.from_numpy(raw.reshape(-1)).to(cuda), n, k)
    return ops.dequantize_gguf(p), lambda x, o: ops.gemm_gguf(x, p, o), ops.gemv_gguf_batched, p


# k: fewer 64-wide chunks than the workgroup's eight waves, and 18 chunks (some waves one more)
@pytest.mark.parametrize("fmt,k", [("int4_32", 192), ("int4_64", 192), ("int4_64", 1152), ("int4_128", 1152),
                                   ("int4_256", 1280), ("int8_channel", 192), ("int8_tensor", 1152),
                                   ("q4_0", 1152), ("q8_0", 192), ("q8_0", 1152), ("nf4_64", 256), ("nf4_128", 1152)])
@pytest.mark.parametrize("m,n", SHAPES)
def test_split_vs_float64(cuda, fmt, k, m, n):
    wd, run, run_batched = _weight(fmt, n, k, cuda)
    x = torch.from_numpy(synth.activations_bf16(33, m, m, k).view(np.int16)).view(torch.bfloat16).to(cuda)
    x64, w64 = x.cpu().double(), wd.cpu().double()
    ref, mag = x64 @ w64.t(), x64.abs() @ w64.abs().t()
    # f32 roundings on a path of one product: an MFMA step every 16 of K, a scale every 32, the sum of
    # eight waves and the dequantized weight's own; each at most 2^-24 of the magnitudes summed
    bound = (k / 16 + k / 32 + 10) * 2.0 ** -24 * mag
    if fmt.startswith("nf4"):  # two MFMAs a step; T_hi + T_lo is within 2^-17 of the table value
        bound += (k / 16 * 2.0 ** -24 + 2.0 ** -17) * mag
    y = run(x, torch.float32)
    assert bool(((y.cpu().double() - ref).abs() <= bound).all()), (fmt, m, n, k)
    yb = run(x, torch.bfloat16)
    assert torch.equal(yb, y.to(torch.bfloat16))
    # (batched INT4 takes groups of 128; a single GGUF call of two rows runs the M = 1 kernel)
    if m <= 64 and (fmt in ("int4_128", "int8_channel", "int8_tensor") or fmt[0] == "n" or m > 2 and fmt[0] == "q"):
        yy = torch.empty_like(y)
        run_batched(x, yy)  # one problem: by the same rule as the single call
        assert torch.equal(yy, y)


# the seven projections of a decoder layer in n, short in k, two with remainders: more than three 32 x 32
# tiles per CU, so that M <= 32 runs 64 (n) x 32 tiles where the format has them
LAYER = [(4096, 256)] * 3 + [(4099, 384), (11008, 256), (11001, 256), (4096, 1152)]


@pytest.mark.parametrize("fmt", ["int4_128", "int8_channel", "int8_tensor", "nf4_64", "q4_0", "q8_0"])
def test_layer_batch_gives_single_call_bits(cuda, fmt):
    """A problem's bits do not depend on what else is in its batch: the seven matrices of a layer in one
    launch give the bits of one call each, which are within the float64 bound."""
    made = [_packed(fmt, n, k, cuda) for n, k in LAYER]
    run_batch, ps = made[0][2], [p for *_, p in made]
    for m in (2, 4, 8, 16, 17, 24, 32, 33, 40, 64):
        xs = [torch.from_numpy(synth.activations_bf16(36 + i, m, m, k).view(np.int16)).view(torch.bfloat16).to(cuda)
              for i, (_, k) in enumerate(LAYER)]
        ys = [torch.full((m, n), float("nan"), device=cuda) for n, _ in LAYER]
        run_batch(xs, ps, ys)
        for i, ((n, k), (wd, run, _, _)) in enumerate(zip(LAYER, made)):
            # (a single GGUF call of two rows runs the M = 1 kernel)
            assert m == 2 and fmt[0] == "q" or torch.equal(ys[i], run(xs[i], torch.float32)), (fmt, m, i)
            x64, w64 = xs[i].double(), wd.double()
            # as in test_split_vs_float64; the kernels of up to 32 rows round at most twice as often (f16
            # products, a power-of-two scale per 128)
            bound = 2 * (k / 16 + k / 32 + 10) * 2.0 ** -24 * (x64.abs() @ w64.abs().t())
            if fmt.startswith("nf4"):
                bound += (k / 16 * 2.0 ** -24 + 2.0 ** -17) * (x64.abs() @ w64.abs().t())
            assert bool(((ys[i].double() - x64 @ w64.t()).abs() <= bound).all()), (fmt, m, i)


# (m, n): one round of 96-row tiles against one or two of 128; two rounds of 128-row tiles against one
# of 256 (INT8)
@pytest.mark.parametrize("fmt", ["int4_128", "int8_channel", "q4_0", "q8_0"])
@pytest.mark.parametrize("m,n", [(97, 300), (1536, 5376), (1601, 5377)])
def test_prefill_tile_heights_vs_float64(cuda, fmt, m, n, monkeypatch):
    """The one-MFMA prefill kernel at each of its tile heights (96, 128, 256 rows by rounds over the
    CUs), row and column remainders included."""
    monkeypatch.setenv("CASTFORGE_PREFILL_I4", "1")
    k = 256
    wd, run, _ = _weight(fmt, n, k, cuda)
    x = torch.from_numpy(synth.activations_bf16(35, m, m, k).view(np.int16)).view(torch.bfloat16).to(cuda)
    ref, mag = x.double() @ wd.double().t(), x.double().abs() @ wd.double().abs().t()
    bound = (k / 16 + k / 32 + 10) * 2.0 ** -24 * mag
    y = run(x, torch.float32)
    assert bool(((y.double() - ref).abs() <= bound).all()), (fmt, m, n)


@pytest.mark.parametrize("m", [2, 9, 16, 24, 40, 64])
def test_batch_over_two_kernels(cuda, m):
    """A problem with more groups in a row than the K-split kernel takes runs on the skinny kernel, the others
    of its batch on the K-split kernel: each gives the bits of its single call."""
    made = [_packed("int4_128", n, k, cuda) for n, k in [(97, 1152), (70, 16640), (33, 256)]]
    xs = [torch.from_numpy(synth.activations_bf16(39 + i, m, m, wd.shape[1]).view(np.int16)).view(torch.bfloat16).to(cuda)
          for i, (wd, *_) in enumerate(made)]
    ys = [torch.full((m, wd.shape[0]), float("nan"), device=cuda) for wd, *_ in made]
    ops.gemv_w4a16_batched(xs, [p for *_, p in made], ys)
    for x, y, (wd, run, _, _) in zip(xs, ys, made):
        assert torch.equal(y, run(x, torch.float32))
        x64, w64, k = x.double(), wd.double(), wd.shape[1]
        bound = 2 * (k / 16 + k / 32 + 10) * 2.0 ** -24 * (x64.abs() @ w64.abs().t())
        assert bool(((y.double() - x64 @ w64.t()).abs() <= bound).all()), (m, k)


def _at_end(t):
    """A copy of t in the last bytes of a 32 MiB allocation of its own."""
    b = t.contiguous().reshape(-1).view(torch.uint8)
    buf = torch.empty(32 << 20, dtype=torch.uint8, device=t.device)
    buf[-b.numel():] = b
    return buf[-b.numel():].view(t.dtype).reshape(t.shape)


@pytest.mark.parametrize("fmt", ["int4_128", "int4_32", "int8_channel", "q4_0", "q8_0", "nf4_64"])
@pytest.mark.parametrize("prefill", [False, True])
def test_operands_at_the_end_of_their_allocation(cuda, fmt, prefill, monkeypatch):
    """Rows past M and N are not read: x and the codes end where their allocation ends, with tiles of every
    kernel that hold few rows, and the results are the bits of the same operands elsewhere."""
    if prefill:
        monkeypatch.setenv("CASTFORGE_PREFILL_I4", "1")
    k, n = 1152, 97
    _, run, _, p = _packed(fmt, n, k, cuda)
    codes = p[0] if isinstance(p, tuple) else p.codes
    end = (_at_end(codes), p[1]) if isinstance(p, tuple) else type(p)(**{**vars(p), "codes": _at_end(codes)})
    if isinstance(p, tuple):
        run_end = lambda x, o: ops.gemm_w8a16(x, *end, fmt[5:], o)  # noqa: E731
    else:
        call = ops.gemm_w4a16 if fmt[0] == "i" else ops.gemm_nf4 if fmt[0] == "n" else ops.gemm_gguf
        run_end = lambda x, o: call(x, end, o)  # noqa: E731
    for m in (3, 17, 33, 65, 130, 2050):
        x = torch.from_numpy(synth.activations_bf16(38, m, m, k).view(np.int16)).view(torch.bfloat16).to(cuda)
        assert torch.equal(run_end(_at_end(x), torch.float32), run(x, torch.float32)), (fmt, m)
