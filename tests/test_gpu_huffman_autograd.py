"""Inputs that ask for gradients through the batched Huffman linear: the
products are not differentiable; which outputs carry a graph is the same for
every route of a token count."""
import numpy as np
import pytest
import torch

import codebook_builder as cbb
import huffman_codebook as hc
from conftest import rel_l2
from test_gpu_huffman import _lin

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,K,dtype,graph", [
    (32, 2048, torch.float32, True),        # the few-token operator
    (20, 2048, torch.bfloat16, True),
    (33, 2048, torch.float32, False), (33, 2048, torch.bfloat16, False),
    (70, 4096, torch.float32, False), (70, 4096, torch.bfloat16, False),
    (20, 9216, torch.float32, False), (20, 9216, torch.bfloat16, False)])
def test_outputs_of_inputs_with_gradients(cuda, T, K, dtype, graph):
    M = 8
    w = cbb.bf16_round(np.random.default_rng(T + K).standard_normal((M, K)) * 0.02)
    cb, idx = cbb.frequency_sorted_codebook(w)
    lin = _lin(hc.huffman_encode_indices(idx, shape=(M, K)), cb, M, K)
    assert lin.split is not None
    x = torch.randn(T, K, device=cuda).to(dtype).requires_grad_()
    y = lin(x)
    assert y.dtype == dtype and y.requires_grad == graph
    ref = x.detach().double().cpu().numpy() @ w.astype(np.float64).T
    assert rel_l2(y.detach().double().cpu().numpy(), ref) <= (1e-6 if dtype == torch.float32 else
                                                             2.0 ** -9)
