"""The batched fixed-width linear by workspace size and codebook kind: which
kernel a call gets, and that every one gives the product of the decoded
matrix (float64 of the same values)."""
import pytest
import torch

import cbq_native as nat
from test_gpu_frag_gemm import TOL_F32, _matrix, _rel

pytestmark = pytest.mark.gpu
# one fp32 rounding per product and addition of a chain of K / S, random signs
TOL_CHAIN = 1e-6


def _f32_ws(cuda, x, packed, cb, M, K, bits, n):
    lib = nat.load()
    ws = torch.full((max(n, 16),), 0xFF, dtype=torch.uint8, device=cuda)
    guard = torch.full((4096,), 0xA5, dtype=torch.uint8, device=cuda)
    buf = torch.cat([ws, guard])
    out = torch.full((x.shape[0], M), float("nan"), device=cuda)
    nat.check(lib.cbq_linear_f32_ws(x.data_ptr(), packed.data_ptr(), cb.data_ptr(),
                                    out.data_ptr(), x.shape[0], M, K, cb.numel(), bits,
                                    buf.data_ptr(), n, nat.stream_ptr(cuda)), "cbq_linear_f32_ws")
    assert torch.equal(buf[ws.numel():], guard)          # nothing past the workspace
    return out


@pytest.mark.parametrize("T,M,K,bits", [(64, 128, 4096, 13), (300, 200, 2048, 8),
                                        (513, 136, 2080, 11)])
def test_f32_split_k_below_the_gemm_workspace(cuda, T, M, K, bits):
    """A workspace one byte short of the decode-first GEMM's that holds the
    fp32 kernel's partials: K is split there, so sums round differently from
    ck_linear_f32's single chain."""
    print(f"split K T{T} M{M} K{K} bits{bits}", flush=True)
    lib = nat.load()
    packed, cb, w = _matrix(cuda, M, K, bits, "bf16", T + M)
    x = torch.randn(T, K, device=cuda, generator=torch.Generator(device="cuda").manual_seed(K))
    ref = x.double() @ w.T
    n = int(lib.cbq_linear_f32_workspace(T, M, K))
    one = torch.empty(T, M, device=cuda)
    nat.check(lib.ck_linear_f32(x.data_ptr(), packed.data_ptr(), cb.data_ptr(), one.data_ptr(), T,
                                M, K, cb.numel(), bits, nat.stream_ptr(cuda)), "ck_linear_f32")
    y = _f32_ws(cuda, x, packed, cb, M, K, bits, n - 1)
    assert _rel(y, ref) <= TOL_CHAIN and not torch.equal(y, one)
    assert torch.equal(_f32_ws(cuda, x, packed, cb, M, K, bits, 16), one)   # no room: one chain
    assert _rel(_f32_ws(cuda, x, packed, cb, M, K, bits, n), ref) <= TOL_F32


def _indices(packed, M, K, bits):
    """The stream's indices, unpacked bit by bit."""
    b = packed[:M * K * bits // 8, None].to(torch.int64) >> torch.arange(8, device=packed.device)
    b = (b & 1).reshape(M * K, bits)
    return (b << torch.arange(bits, device=packed.device)).sum(1).reshape(M, K)


def _layer(packed, cb, M, K, bits):
    from device_formats import FixedTensor
    from gpu_accelerated_functions import GPUAcceleratedLinear
    return GPUAcceleratedLinear.from_device("w", FixedTensor("w", (M, K), bits, "x", packed, cb))


def _us(fn):
    fn()
    e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
    e[0].record()
    for _ in range(3):
        fn()
    e[1].record()
    torch.cuda.synchronize()
    return e[0].elapsed_time(e[1]) / 3e-3


@pytest.mark.parametrize("T,M,K,bits", [(33, 130, 96, 13), (40, 1024, 2048, 14), (64, 4096, 512, 13),
                                        (70, 200, 4096, 8), (300, 1030, 2048, 12)])
@pytest.mark.parametrize("declared", [True, False])
def test_non_finite_codebook_keeps_its_rate(cuda, T, M, K, bits, declared):
    """One infinity in the codebook: infinities and NaNs where the products
    have them, with the kind the module found at load (the fp32 kernel) and
    with none (the GEMM's own fp32 products); no more than ten times the time
    of a finite codebook (one output at a time took 300 times)."""
    from gpu_accelerated_functions import cbq_ops
    print(f"non-finite T{T} M{M} K{K} bits{bits} declared {declared}", flush=True)
    packed, cb, w = _matrix(cuda, M, K, bits, "inf", T + M)
    x = torch.randn(T, K, device=cuda, generator=torch.Generator(device="cuda").manual_seed(K))
    x[5] = x[5].bfloat16().float()                       # zero lower parts
    x[7, ::3] = 0.0
    x[9, 1] = float("-inf")
    layer = _layer(packed, cb, M, K, bits)
    assert layer.cb_kind == cbq_ops.CB_NON_FINITE
    if not declared:
        layer.cb_kind = cbq_ops.CB_UNKNOWN
    y, ref = layer(x), x.double() @ w.T
    assert torch.equal(y.isnan(), ref.isnan())
    assert torch.equal(y.isposinf(), ref.isposinf()) and torch.equal(y.isneginf(), ref.isneginf())
    ok = ref.isfinite()
    if bool(ok.any()):
        assert _rel(y[ok], ref[ok]) <= TOL_CHAIN
    plain = _layer(packed, torch.where(cb.isfinite(), cb, 0.01), M, K, bits)
    assert _us(lambda: layer(x)) <= 10 * _us(lambda: plain(x)) + 50


def test_codebook_changed_in_place(cuda):
    """The kind is a hint: a codebook written after the module was made gives
    its own product, whatever it then holds."""
    T, M, K, bits = 80, 320, 1024, 10
    packed, cb, w = _matrix(cuda, M, K, bits, "bf16", 11)
    x = torch.randn(T, K, device=cuda, generator=torch.Generator(device="cuda").manual_seed(2))
    layer = _layer(packed, cb, M, K, bits)
    assert _rel(layer(x), x.double() @ w.T) <= TOL_F32
    g = torch.Generator(device="cuda").manual_seed(3)
    for fill in ("fp32", "inf", "bf16"):
        new = torch.randn(cb.numel(), device=cuda, generator=g) * 0.05
        if fill != "fp32":
            new = new.bfloat16().float()
        if fill == "inf":
            new[3] = float("inf")
        idx = _indices(packed, M, K, bits).clamp_max(cb.numel() - 1)
        cb.copy_(new)
        ref = x.double() @ cb[idx].double().T
        for xx in (x, x.bfloat16()):
            r = ref if xx is x else xx.double() @ cb[idx].double().T
            y = layer(xx)
            if xx is not x and fill == "inf":
                continue                                # (bf16 x: hi + lo parts, as ever)
            assert torch.equal(y.isnan(), r.isnan())
            ok = r.isfinite()
            if bool(ok.any()):
                assert _rel(y[ok], r[ok]) <= (TOL_CHAIN if xx is x else 2.0 ** -9)


def _gemm(cuda, x, packed, cb, M, K, bits, kind):
    lib = nat.load()
    T, bf16 = x.shape[0], int(x.dtype == torch.bfloat16)
    n = int(lib.cbq_linear_gemm_workspace(T, M, K, bits, bf16, kind))
    buf = torch.full((max(n, 16) + 4096,), 0xA5, dtype=torch.uint8, device=cuda)
    out = torch.full((T, M), float("nan"), dtype=x.dtype, device=cuda)
    nat.check(lib.cbq_linear_gemm(x.data_ptr(), bf16, packed.data_ptr(), cb.data_ptr(),
                                  out.data_ptr(), T, M, K, cb.numel(), bits, kind, buf.data_ptr(),
                                  n, nat.stream_ptr(cuda)), "cbq_linear_gemm")
    assert bool((buf[max(n, 16):] == 0xA5).all())        # nothing past the workspace
    return out


@pytest.mark.parametrize("T,M,K,bits", [(64, 33, 64, 12), (33, 4100, 1056, 13), (300, 520, 4096, 8),
                                        (129, 2049, 96, 14), (700, 1030, 544, 11),
                                        (1030, 3000, 544, 13), (2050, 4000, 1024, 10)])
@pytest.mark.parametrize("kind", [0, 1, 2, 3])
@pytest.mark.parametrize("holds", ["bf16", "fp32"])
def test_every_kind_gives_the_product(cuda, T, M, K, bits, kind, holds):
    """Declared as anything, a codebook's product is its own: one part of the
    weights reserved where three are needed falls back to fp32 products."""
    print(f"kind {kind} {holds} T{T} M{M} K{K} bits{bits}", flush=True)
    packed, cb, w = _matrix(cuda, M, K, bits, holds, T + M)
    x = torch.randn(T, K, device=cuda, generator=torch.Generator(device="cuda").manual_seed(K))
    assert _rel(_gemm(cuda, x, packed, cb, M, K, bits, kind), x.double() @ w.T) <= TOL_CHAIN
    xb = x.bfloat16()
    assert _rel(_gemm(cuda, xb, packed, cb, M, K, bits, kind), xb.double() @ w.T) <= 2.0 ** -9


@pytest.mark.parametrize("dtype,K,kind,holds", [
    (torch.bfloat16, 524320, 0, "fp32"), (torch.bfloat16, 524320, 1, "bf16"),
    (torch.float32, 262176, 0, "fp32"), (torch.float32, 262176, 1, "fp32"),
    (torch.float32, 786464, 1, "bf16")])
def test_slabs(cuda, dtype, K, kind, holds):
    """Rows so long that the weights go slab by slab (256 rows each at least):
    two and three parts of the weights, one, and the fp32 products of a
    codebook declared to need one."""
    T, M, bits = 80, 520, 12
    print(f"slabs {dtype} K{K} kind {kind} {holds}", flush=True)
    packed, cb, w = _matrix(cuda, M, K, bits, holds, 3)
    x = torch.randn(T, K, device=cuda).to(dtype)
    y, ref = _gemm(cuda, x, packed, cb, M, K, bits, kind), x.double() @ w.T
    if dtype == torch.bfloat16:
        assert _rel(y, ref) <= 2.0 ** -9
    else:
        # A sum of n terms of random sign in one chain of roundings, each half
        # an ulp (2^-24) of a partial sum that grows as the root of its length:
        # rel-L2 <= 2^-24 sqrt(n / 2).  Fragments: a chain of 16 groups x 3 (6
        # with three parts of W) MFMAs, then one of K / 512 totals; fp32
        # products: one of K / 4 MFMAs.  (No more where K is split.)
        n = 48 * (2 if holds == "fp32" else 1) + K / 512
        if kind == 1 and holds == "fp32":
            n = K / 4
        assert _rel(y, ref) <= 2.0 ** -24 * (n / 2) ** 0.5


@pytest.mark.parametrize("M,K", [(200704, 1024), (66000, 3072), (49300, 4096)])
def test_split_slabs(cuda, M, K):
    """Split-format matrices of more than 384 MiB of fragments: the second
    slab's rows start inside the matrix, in each chunk geometry (whole rows
    per chunk, chunks across rows, whole chunks per row)."""
    import cbq_ops
    from test_gpu_frag_gemm import _split_matrix
    print(f"split slabs M{M} K{K}", flush=True)
    assert 2 * M * K > 384 << 20
    t, w = _split_matrix(cuda, M, K, 5)
    x = torch.randn(33, K, device=cuda)
    op = cbq_ops.load().split_gemm
    y, ref = op(x, *t.keep, M), x.double() @ w.T
    assert _rel(y, ref) <= TOL_F32
    rows = (y.double() - ref).norm(dim=0) / ref.norm(dim=0)    # every row, both slabs
    assert float(rows.max()) <= 10 * TOL_F32
    yb = op(x.bfloat16(), *t.keep, M)
    assert _rel(yb, x.bfloat16().double() @ w.T) <= 2.0 ** -9


@pytest.mark.parametrize("kind", [0, 1])
def test_bf16_non_finite_x(cuda, kind):
    """Infinities and NaNs of bf16 x over a lossless codebook."""
    T, M, K, bits = 300, 1040, 2048, 13
    packed, cb, w = _matrix(cuda, M, K, bits, "bf16", 5)
    x = torch.randn(T, K, device=cuda).bfloat16()
    x[3, 7], x[9, 100], x[11, 0] = float("inf"), float("-inf"), float("nan")
    x[20] = 0.0
    assert nat.load().cbq_linear_gemm_workspace(T, M, K, bits, 1, kind) > 0
    y, ref = _gemm(cuda, x, packed, cb, M, K, bits, kind), x.double() @ w.T
    assert torch.equal(y.isnan(), ref.isnan())
    assert torch.equal(y.isposinf(), ref.isposinf()) and torch.equal(y.isneginf(), ref.isneginf())
    ok = ref.isfinite()
    assert _rel(y[ok], ref[ok]) <= 2.0 ** -9


def test_huffman_non_finite_codebook(cuda):
    """A Huffman matrix with an infinite value, batched: infinities and NaNs
    where the products have them, in both formats."""
    import numpy as np
    import codebook_builder as cbb
    import huffman_codebook as hc
    from test_gpu_huffman import _lin
    M, K = 64, 1024
    rng = np.random.default_rng(3)
    wn = cbb.bf16_round(rng.standard_normal((M, K)) * 0.02)
    cb, idx = cbb.frequency_sorted_codebook(wn)
    cb = cb.copy()
    cb[len(cb) // 2] = np.inf
    enc = hc.huffman_encode_indices(idx, shape=(M, K))
    w = torch.from_numpy(cb).to(cuda)[torch.from_numpy(idx.astype(np.int64)).to(cuda)]
    w = w.reshape(M, K).double()
    for layout in ("auto", "stream"):
        lin = _lin(enc, cb, M, K, layout=layout)
        for T in (64, 100):
            x = torch.randn(T, K, device=cuda)
            x[1] = x[1].bfloat16().float()
            y, ref = lin(x), x.double() @ w.T
            assert torch.equal(y.isnan(), ref.isnan()), (layout, T)
            assert torch.equal(y.isposinf(), ref.isposinf())
            ok = ref.isfinite()
            assert _rel(y[ok], ref[ok]) <= TOL_CHAIN


@pytest.mark.parametrize("K", [32, 64, 128, 256, 1024, 8192])
@pytest.mark.parametrize("kind", [0, 2])
@pytest.mark.parametrize("one_sign", [False, True])
def test_fp32_codebook_no_further_off_than_fp32_products(cuda, K, kind, one_sign):
    """A k-means codebook under fp32 x: the error against 64 bits is no larger
    than that of ck_linear_f32's exact products in one chain (5% for the
    chance of these values)."""
    T, M, bits = 512, 1024, 8
    packed, cb, _ = _matrix(cuda, M, K, bits, "fp32", K)
    x = torch.randn(T, K, device=cuda, generator=torch.Generator(device="cuda").manual_seed(K))
    if one_sign:
        cb, x = cb.abs(), x.abs()
    ref = x.double() @ cb[_indices(packed, M, K, bits).clamp_max(cb.numel() - 1)].double().T
    one = torch.empty(T, M, device=cuda)
    lib = nat.load()
    nat.check(lib.ck_linear_f32(x.data_ptr(), packed.data_ptr(), cb.data_ptr(), one.data_ptr(), T,
                                M, K, cb.numel(), bits, nat.stream_ptr(cuda)), "ck_linear_f32")
    y = _gemm(cuda, x, packed, cb, M, K, bits, kind)
    assert _rel(y, ref) <= 1.05 * _rel(one, ref)
