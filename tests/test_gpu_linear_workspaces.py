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
