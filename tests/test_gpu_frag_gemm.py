"""The decode-first batched GEMM (cbq_linear_f32_ws with its workspace) at the
edges of its tiles, column groups, K splits, slabs and codebook kinds, against
float64 products of the decoded matrix.

Bound for fp32 x: every product is exact (codebooks of bf16 numbers) or short
of the whole by less than 2^-22 (others), and the sum is rounded to fp32 in
chains of at most 48 MFMAs (96 with three parts of W), whose totals are added
K / 128, K / 256 or K / 512 times (folds of 4, 8 and 16 column groups: below 96
groups, below 400, above): rel-L2 <= 5e-7 for random signs."""
import numpy as np
import pytest
import torch

import cbq_native as nat
import codebook_builder as cbb

pytestmark = pytest.mark.gpu
TOL_F32 = 5e-7


def _matrix(cuda, M, K, bits, kind, seed):
    """(packed, codebook, dense float64 W): indices over the whole width, so
    some lie past C and clamp."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    C = max(2, (1 << bits) * 5 // 8)
    cb = torch.randn(C, device=cuda, generator=g) * 0.02
    if kind != "fp32":
        cb = cb.bfloat16().float()
    if kind == "inf":
        cb[C // 2] = float("inf")
    idx = torch.randint(0, 1 << bits, (M, K), device=cuda, generator=g)
    pk = cbb.pack_torch(idx, bits)
    packed = torch.zeros((pk.numel() + 15) // 16 * 16 + 16, dtype=torch.uint8, device=cuda)
    packed[:pk.numel()] = pk
    return packed, cb, cb[idx.clamp_max(C - 1)].double()


def _run_f32(cuda, x, packed, cb, M, K, bits):
    lib = nat.load()
    T = x.shape[0]
    n = int(lib.cbq_linear_f32_workspace(T, M, K))
    assert n > 0
    ws = torch.full((n,), 0xFF, dtype=torch.uint8, device=cuda)
    out = torch.full((T, M), float("nan"), device=cuda)
    nat.check(lib.cbq_linear_f32_ws(x.data_ptr(), packed.data_ptr(), cb.data_ptr(),
                                    out.data_ptr(), T, M, K, cb.numel(), bits, ws.data_ptr(), n,
                                    nat.stream_ptr(cuda)), "cbq_linear_f32_ws")
    return out


def _run_bf16(cuda, x, packed, cb, M, K, bits):
    lib = nat.load()
    T = x.shape[0]
    n = int(lib.cbq_linear_bf16_gemm_workspace(T, M, K, bits))
    ws = torch.full((max(n, 16),), 0xFF, dtype=torch.uint8, device=cuda)
    out = torch.full((T, M), float("nan"), dtype=torch.bfloat16, device=cuda)
    nat.check(lib.cbq_linear_bf16_ws(x.data_ptr(), packed.data_ptr(), cb.data_ptr(),
                                     out.data_ptr(), T, M, K, cb.numel(), bits, ws.data_ptr(), n,
                                     nat.stream_ptr(cuda)), "cbq_linear_bf16_ws")
    return out


def _rel(y, ref):
    return float((y.double() - ref).norm() / ref.norm())


@pytest.mark.parametrize("T,M,K,bits", [
    (64, 1, 32, 13),            # one column group, one row
    (17, 33, 128, 13), (32, 1000, 4224, 14), (24, 520, 2048, 16),   # few tokens, x as fragments
    (16, 40, 12288, 13), (10, 4100, 12416, 10), (29, 24600, 256, 8),
    (33, 4096, 2048, 13), (48, 31, 96, 12),
    (65, 33, 64, 12),           # a row past a superblock, a token past a tile
    (127, 257, 96, 14), (129, 300, 4064, 13), (192, 520, 288, 11), (257, 1000, 1056, 10),
    (64, 4096, 4096, 13), (300, 2048, 2080, 8), (1030, 3000, 544, 13)])
@pytest.mark.parametrize("kind", ["bf16", "fp32"])
def test_f32_edges(cuda, T, M, K, bits, kind):
    print(f"f32 {kind} T{T} M{M} K{K} bits{bits}", flush=True)
    packed, cb, w = _matrix(cuda, M, K, bits, kind, T + M)
    x = torch.randn(T, K, device=cuda, generator=torch.Generator(device="cuda").manual_seed(K))
    y = _run_f32(cuda, x, packed, cb, M, K, bits)
    assert _rel(y, x.double() @ w.T) <= TOL_F32


def test_f32_slabs(cuda):
    """A row so long that the fragments are written slab by slab."""
    T, M, K, bits = 64, 520, 262176, 12
    packed, cb, w = _matrix(cuda, M, K, bits, "bf16", 3)
    x = torch.randn(T, K, device=cuda)
    assert _rel(_run_f32(cuda, x, packed, cb, M, K, bits), x.double() @ w.T) <= TOL_F32


@pytest.mark.parametrize("kind", ["bf16", "fp32", "inf"])
def test_f32_non_finite(cuda, kind):
    """Infinities and NaNs of x and the codebook reach the outputs that a
    plain fp32 sum gives them."""
    T, M, K, bits = 70, 200, 256, 8
    packed, cb, w = _matrix(cuda, M, K, bits, kind, 5)
    x = torch.randn(T, K, device=cuda)
    x[3, 7], x[9, 100], x[11, 0] = float("inf"), float("-inf"), float("nan")
    x[20] = 0.0
    y = _run_f32(cuda, x, packed, cb, M, K, bits)
    ref = x.double() @ w.T
    assert torch.equal(y.isnan(), ref.isnan())
    assert torch.equal(y.isposinf(), ref.isposinf()) and torch.equal(y.isneginf(), ref.isneginf())
    ok = ref.isfinite()
    assert _rel(y[ok], ref[ok]) <= TOL_F32


def test_f32_scales(cuda):
    """Token rows over 60 decades keep their relative error."""
    T, M, K, bits = 64, 96, 512, 13
    packed, cb, w = _matrix(cuda, M, K, bits, "bf16", 6)
    s = 10.0 ** torch.linspace(-30, 30, T, device=cuda, dtype=torch.float64)
    x = (torch.randn(T, K, device=cuda).double() * s[:, None]).float()
    y, ref = _run_f32(cuda, x, packed, cb, M, K, bits), x.double() @ w.T
    assert float(((y.double() - ref).norm(dim=1) / ref.norm(dim=1)).max()) <= 2 * TOL_F32


def test_f32_graph(cuda):
    """Captured and replayed with other inputs in between: the eager result."""
    T, M, K, bits = 100, 1024, 2048, 13
    packed, cb, w = _matrix(cuda, M, K, bits, "bf16", 7)
    lib = nat.load()
    x = torch.randn(T, K, device=cuda)
    n = int(lib.cbq_linear_f32_workspace(T, M, K))
    ws = torch.empty(n, dtype=torch.uint8, device=cuda)
    out = torch.empty(T, M, device=cuda)

    def call():
        nat.check(lib.cbq_linear_f32_ws(x.data_ptr(), packed.data_ptr(), cb.data_ptr(),
                                        out.data_ptr(), T, M, K, cb.numel(), bits, ws.data_ptr(),
                                        n, nat.stream_ptr(cuda)), "cbq_linear_f32_ws")
    call()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for i in range(3):
        x.copy_(torch.randn(T, K, device=cuda))
        eager = _run_f32(cuda, x, packed, cb, M, K, bits)
        graph.replay()
        assert torch.equal(out, eager)


@pytest.mark.parametrize("T,M,K,bits", [
    (17, 33, 128, 13), (32, 1000, 4224, 14), (33, 16, 256, 12), (48, 300, 1152, 13),
    (49, 12288, 128, 10), (64, 520, 2048, 16), (64, 4100, 1024, 13),     # few-token kernel
    (63, 70, 96, 13),                                                    # refused by it
    (16, 70, 20480, 12), (30, 1000, 12288, 13), (64, 300, 12288, 14),    # x as fragments
    (65, 33, 64, 12), (127, 257, 96, 14), (129, 300, 4064, 13), (257, 1000, 1056, 10),
    (300, 2048, 2080, 8), (700, 1030, 544, 11), (1030, 3000, 544, 13), (2050, 520, 96, 13)])
@pytest.mark.parametrize("kind", ["bf16", "fp32"])
def test_bf16_edges(cuda, T, M, K, bits, kind):
    """bf16 x: within the rounding of a bf16 output (2^-9 at most, 1.7e-3 in
    the 2-norm for random values)."""
    print(f"bf16 {kind} T{T} M{M} K{K} bits{bits}", flush=True)
    packed, cb, w = _matrix(cuda, M, K, bits, kind, T + M)
    g = torch.Generator(device="cuda").manual_seed(K)
    x = torch.randn(T, K, device=cuda, generator=g).bfloat16()
    y, ref = _run_bf16(cuda, x, packed, cb, M, K, bits), x.double() @ w.T
    assert _rel(y, ref) <= 2.0 ** -9
    # against one rounding of the exact value: at most one step apart
    near = ref.bfloat16().double()
    assert float(((y.double() - near).abs() <= 2.0 ** -7 * near.abs() + 1e-30).double().mean()) > 0.99


def _split_matrix(cuda, M, K, seed):
    import device_formats as dfm
    g = torch.Generator(device="cuda").manual_seed(seed)
    w = (torch.randn(M, K, device=cuda, generator=g) * 0.02).bfloat16()
    cb, lut = cbb.codebook_from_counts_torch(cbb.counts_torch(w))
    idx = lut[cbb.patterns_torch(w).reshape(-1).to(torch.int64)]
    t = dfm.to_split(dfm.encode_huffman("w", idx, cb, (M, K), "mlp_ffn"), idx)
    assert t is not None
    return t, w.double()


@pytest.mark.parametrize("T,M,K", [
    (17, 4, 1024), (33, 100, 1024), (64, 2, 2048), (40, 300, 2048), (130, 132, 3072),
    (17, 1, 4096), (64, 33, 4096), (300, 520, 4096), (20, 68, 5120), (50, 258, 6144),
    (96, 40, 7168), (70, 37, 8192), (18, 132, 9216), (1, 64, 2048)])
def test_split_gemm(cuda, T, M, K):
    """Split-format matrices of every chunk geometry (rows of whole chunks,
    chunks of whole rows, chunks across rows), rows off every tile: fp32 and
    bf16 x."""
    import cbq_ops
    print(f"split T{T} M{M} K{K}", flush=True)
    t, w = _split_matrix(cuda, M, K, M + K)
    x = torch.randn(T, K, device=cuda, generator=torch.Generator(device="cuda").manual_seed(T))
    op = cbq_ops.load().split_gemm
    y = op(x, *t.keep, M)
    assert _rel(y, x.double() @ w.T) <= TOL_F32
    xb = x.bfloat16()
    yb, ref = op(xb, *t.keep, M), xb.double() @ w.T
    assert yb.dtype == torch.bfloat16 and _rel(yb, ref) <= 2.0 ** -8 / 3 ** 0.5 * 1.1


@pytest.mark.parametrize("M,K", [(4, 1024), (36, 3072), (40, 4096)])
def test_split_gemm_stacked_parts(cuda, M, K):
    """The parts of two matrices stacked under one shared table: each part's
    product is its own matrix's, bit for bit (the decoded values are)."""
    from gpu_huffman_functions import build_split, split_prefill, stack_split, stacked_parts
    g = torch.Generator(device="cuda").manual_seed(M + K)
    ws = [(torch.randn(M, K, device=cuda, generator=g) * 0.02).bfloat16() for _ in range(2)]
    cb, lut = cbb.codebook_from_counts_torch(cbb.counts_torch(ws[0]) + cbb.counts_torch(ws[1]))
    sps = [build_split(lut[cbb.patterns_torch(w).reshape(-1).to(torch.int64)].to(torch.int32),
                       cb.cpu().numpy(), cuda) for w in ws]
    keep, _, parts = stack_split(sps, cb.cpu().numpy(), [M, M], K, cuda)
    x = torch.randn(33, K, device=cuda, generator=g)
    for own, part, w in zip(sps, stacked_parts(keep, parts), ws):
        y = split_prefill(part, None, x, M, K, cb, finite=True)
        assert torch.equal(y, split_prefill(own, None, x, M, K, cb, finite=True))
        assert _rel(y, x.double() @ w.double().T) <= TOL_F32


def test_split_gemm_refuses(cuda):
    import cbq_ops
    t, _ = _split_matrix(cuda, 4, 1024, 1)
    op = cbq_ops.load().split_gemm
    with pytest.raises(RuntimeError):
        op(torch.zeros(20, 512, device=cuda), *t.keep, 8)
    with pytest.raises(RuntimeError):
        op(torch.zeros(20, 1024, device=cuda, dtype=torch.float16), *t.keep, 4)


def test_split_module_views_and_types(cuda):
    """The module over strided, misaligned and float16 x equals its result on
    a fresh contiguous copy."""
    from compressed_modules import AdaptiveCodebookLinear
    t, w = _split_matrix(cuda, 64, 2048, 9)
    layer = AdaptiveCodebookLinear.from_device("w", t)
    base = torch.randn(40 * 2048 + 1, device=cuda)
    odd = base[1:].view(40, 2048)                       # 4-byte aligned
    assert torch.equal(layer(odd), layer(odd.clone()))
    tr = torch.randn(2048, 40, device=cuda).t()         # column-major
    assert torch.equal(layer(tr), layer(tr.contiguous()))
    h = torch.randn(2, 20, 2048, device=cuda).half()
    y = layer(h)
    assert y.dtype == torch.float16 and y.shape == (2, 20, 64)
    assert _rel(y.reshape(40, 64), h.reshape(40, 2048).double() @ w.T) <= 2.0 ** -11
