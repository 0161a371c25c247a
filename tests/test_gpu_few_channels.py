"""Mode GEMM whose last step holds at most 16 channels, where the steps go in halves (csrc/layer2d.hip): the kernels with 8 and 16 channels at
the edges of the rule that chooses them, against the oracle, and their operands at any magnitude."""
import numpy as np
import pytest
import torch

import oracle
import turbofno_amd as tf
from conftest import rel_l2
from test_gpu_operand_range import _bound as _range_bound, _cgemm, _worst
from test_gpu_split_products import _bound, _complex, _dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,N,beta", [
    (64, 8, 64, 0.0), (192, 16, 64, 1j),                 # tiles of 16 output channels, a partly filled block
    (8192, 16, 128, 0.5 - 1j),                           # tiles of 32
    (32768 + 64, 8, 192, 0.0), (65536 + 64, 16, 64, 0.0),   # two and less than two blocks per CU
    (131072 + 64, 16, 192, 0.5),                         # more: fp32 matrix instructions
    (163840, 8, 128, 0.0), (163840 + 64, 16, 128, 0.0),  # five, and just above: fp32, persistent
    (524288, 16, 128, 0.0),                              # sixteen: tiles of 128 output channels
    (21120, 16, 192, 0.5), (12800, 8, 320, 0.0), (10624, 16, 384, 0.0),     # one round of 83, 50 and 42 blocks: no groups of eight
    (16384, 104, 128, 0.0), (65536 + 64, 48, 64, 1.0),   # three whole steps and a quarter, one and a half
])
def test_cgemm_with_a_short_last_step(M, K, N, beta):
    print("short step", M, K, N, beta, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(M + K)
    A = torch.view_as_complex(torch.rand((K, M, 2), device="cuda", generator=gen) * 2 - 1)
    W = _complex(np.random.default_rng(M + K + N), N, K) / np.float32(np.sqrt(K))
    C0 = torch.full((N, M), float("nan"), dtype=torch.complex64, device="cuda") if beta == 0.0 else \
        torch.view_as_complex(torch.rand((N, M, 2), device="cuda", generator=gen) * 2 - 1)
    C = C0.clone()
    tf.cgemm(M, N, K, A, _dev(W), C, 0.5 - 0.75j, beta)
    torch.cuda.synchronize()
    assert not bool(torch.isnan(torch.view_as_real(C)).any())
    idx = torch.tensor(sorted({0, 17, M // 2, M - 65, M - 64, M - 1}), device="cuda") if M > 8192 else torch.arange(M, device="cuda")
    pick = lambda a: a.index_select(1, idx).cpu().numpy()
    ref = oracle.cgemm(pick(A), W, 0.5 - 0.75j)
    if beta != 0.0:
        ref = ref + beta * pick(C0).astype(np.complex128)
    assert rel_l2(pick(C), ref) < _bound(K)


@pytest.mark.parametrize("scale", [1e-35, 1e-37, 1e37])
@pytest.mark.parametrize("M,K,N", [(64, 16, 64), (65536 + 64, 8, 64), (32768 + 64, 48, 128), (524288, 16, 128)])
def test_short_steps_of_any_magnitude(M, K, N, scale):
    """a strip of columns of A, then every third row of W, at the given magnitude among others near one"""
    print("short step range", M, K, N, scale, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(M + K)
    A = torch.view_as_complex(torch.rand((K, M, 2), device="cuda", generator=gen) * 2 - 1)
    W = _complex(np.random.default_rng(M + K), N, K) / np.float32(np.sqrt(K))
    C0 = torch.zeros((N, M), dtype=torch.complex64, device="cuda")
    idx = torch.tensor([0, 5, M - 20, M - 1], device="cuda")
    for where in "AW":
        As, Ws = A.clone(), W.copy()
        if where == "A":
            As[:, :16] *= scale
            As[:, M - 32:] *= scale
        else:
            Ws[1::3] *= np.float32(scale)
        got = _cgemm(As, Ws, 0.0, C0).index_select(1, idx).cpu().numpy().astype(np.complex128)
        ref = oracle.cgemm(As.index_select(1, idx).cpu().numpy(), Ws, 1.0)
        # one row holds four values here: single products may differ by twice as much as one fp32 rounding each
        assert _worst(got, ref, 0 if where == "A" else 1) < 2 * _range_bound(K)
