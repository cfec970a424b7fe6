"""cbq_linear_gemm_workspace: what a batched call reserves (host arithmetic, no
GPU needed)."""
import pytest

import cbq_native as nat


@pytest.fixture(scope="module")
def ws():
    lib = nat.load()

    def size(T, M, K, bits, x_bf16=0, kind=0):
        return int(lib.cbq_linear_gemm_workspace(T, M, K, bits, x_bf16, kind))
    return size


@pytest.mark.parametrize("bits", [1, 4, 9, 15, 16])
@pytest.mark.parametrize("x_bf16", [0, 1])
@pytest.mark.parametrize("kind", [0, 1, 2, 3])
def test_refused_widths_reserve_nothing(ws, bits, x_bf16, kind):
    """No prompt kernel takes these widths, so no call may allocate for one
    (16 bits: up to 64 tokens have the few-token kernel's copy of x)."""
    for T in (70, 128, 512, 2048):
        for M, K in ((1024, 2048), (12288, 4096), (4096, 12288)):
            assert ws(T, M, K, bits, x_bf16, kind) == 0, (T, M, K)


@pytest.mark.parametrize("x_bf16", [0, 1])
def test_taken_widths_reserve(ws, x_bf16):
    for bits in (8, 10, 11, 12, 13, 14):
        assert ws(512, 4096, 4096, bits, x_bf16) > 512 * 4096 * 2
        assert ws(1, 4096, 4096, bits, x_bf16) == 0


def test_one_part_of_a_lossless_codebook(ws):
    """A codebook of bf16 numbers reserves two bytes a weight beside x's
    fragments and the partials, one of other values three (fp32 x) or two
    (bf16 x) times that; an unknown one as much as any."""
    M, K, BF16, FP32 = 12288, 4096, 1, 2
    w = 2 * M * K
    for T in (33, 512, 2048):
        assert 2 * w > ws(T, M, K, 13, 0, BF16) > w
        assert ws(T, M, K, 13, 0, FP32) >= 3 * w or T < 300      # (not the GEMM's tokens)
        assert ws(T, M, K, 13, 0, 0) >= max(3 * w, ws(T, M, K, 13, 0, FP32))
    T = 2048                                       # (decodes first)
    assert 2 * w > ws(T, M, K, 13, 1, BF16) > w
    # a lossless lm_head: slabs of at most 384 MiB
    x = 512 * 4096 * 6
    assert ws(512, 151936, 4096, 13, 0, BF16) <= (384 << 20) + x + (1 << 20)


def test_codebook_kind():
    import numpy as np
    import torch
    import cbq_ops as o
    cb = np.array([0.0, -0.0, 1.5, -2.0 ** -126, 2.0 ** -133], np.float32)
    for values, want in (([], o.CB_BF16), ([0.1], o.CB_FP32), ([2.0 ** -140], o.CB_FP32),
                         ([np.inf], o.CB_NON_FINITE), ([0.1, -np.inf], o.CB_NON_FINITE),
                         ([np.nan], o.CB_NON_FINITE)):
        a = np.concatenate([cb, np.array(values, np.float32)])
        assert o.codebook_kind(a) == want == o.codebook_kind(torch.from_numpy(a))


@pytest.mark.parametrize("kind", [0, 1, 2])
def test_64_bf16_tokens_reserve_for_the_few_token_kernel(ws, kind):
    """K % 128 == 0: at most x's fragments."""
    for M, K in ((4096, 4096), (12288, 4096), (4096, 12288)):
        assert ws(64, M, K, 13, 1, kind) <= 64 * K * 2
    assert ws(64, 4096, 4064, 13, 1, kind) > 4096 * 4064      # a prompt kernel's shape


def test_fp32_codebooks_take_the_faster_route(ws):
    """fp32 x over a k-means codebook: token tiles (no workspace), the fp32
    kernel (its split-K partials) or the GEMM (three parts of W), as they were
    measured faster; a lossless codebook takes the GEMM from 33 tokens."""
    BF16, FP32, NON_FINITE = 1, 2, 3

    def route(T, M, K, bits):
        n = ws(T, M, K, bits, 0, FP32)
        if n == 0:
            return "tiles"
        return "gemm" if n >= 6 * M * K else "fp32"

    for T, M, K, bits, want in (
            (33, 4096, 12288, 8, "tiles"), (33, 12288, 4096, 13, "tiles"),
            (33, 4096, 4096, 8, "tiles"), (48, 2048, 1024, 13, "tiles"),
            (63, 1024, 2048, 8, "gemm"), (48, 512, 4064, 8, "gemm"),
            (33, 9000, 4064, 13, "tiles"), (64, 4096, 12288, 8, "fp32"),
            (128, 4096, 12288, 13, "fp32"), (128, 4096, 4096, 13, "fp32"),
            (128, 6144, 2048, 13, "fp32"), (128, 6144, 2048, 8, "gemm"),
            (300, 4096, 12288, 8, "gemm"), (300, 12288, 4096, 13, "gemm"),
            (512, 4096, 4096, 8, "gemm"), (768, 1024, 2048, 13, "gemm")):
        assert route(T, M, K, bits) == want, (T, M, K, bits, ws(T, M, K, bits, 0, FP32))
        assert ws(T, M, K, bits, 0, BF16) > 2 * M * K
