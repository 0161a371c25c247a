"""The 512-thread kernel of small grids (csrc/layer1d_small.hip) at the edges of its rounds, weight tiles and output tiles, against the
oracle; the halves of the layer reach it in test_gpu_split_products.py and test_gpu_operand_range.py."""
import numpy as np
import pytest
import torch

import oracle
import turbofno_amd as tf
from conftest import rel_l2
from test_gpu_operand_range import _layer_check, _x
from test_gpu_split_products import _bound, _complex, _dev

pytestmark = pytest.mark.gpu

# K: half a step; a short last round; more than one tile of weights (WKC = 32 channels with 64 outputs, 64 with 32, 128 with 16)
SHAPES = [(1, 8, 64), (9, 40, 64), (3, 72, 128), (5, 136, 192)]


@pytest.mark.parametrize("DY", [128, 256, 512, 1024])
@pytest.mark.parametrize("S,K,N", SHAPES)
@pytest.mark.parametrize("tile", [64, 32, 16])
def test_small_grid_edges(tile, S, K, N, DY, algo_1d):
    """selector 2: blocks of 64 output channels, 4: of 32 (DY = 128 / 256, else by size); by size: of 16. Every row of y written (y starts as NaN)."""
    print("small grid", tile, S, K, N, DY, flush=True)
    algo_1d({64: 2, 32: 4, 16: 0}[tile])
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        expect = 64 if tile == 64 else 32 if tile == 32 and DY <= 256 else 16
        assert tf.query_1d_tile(DY, S, N, K, compute_units=0) == expect
    x, W = _x(S, DY, K), _complex(np.random.default_rng(S), N, K) / np.float32(np.sqrt(K))
    y = torch.full((N, S, DY), float("nan"), dtype=torch.complex64, device="cuda")
    tf.layer_1d(x, _dev(W), y=y, alpha=0.5 - 0.75j)
    torch.cuda.synchronize()
    assert not bool(torch.isnan(torch.view_as_real(y)).any()), "rows of y left unwritten"
    assert rel_l2(y.cpu().numpy(), oracle.layer_1d(x.cpu().numpy(), W, 0.5 - 0.75j)) < _bound(K, 2)


@pytest.mark.parametrize("scale", [1e-35, 1e-37, 1e20])
@pytest.mark.parametrize("algo,S,DY,K,N", [(0, 3, 128, 40, 64), (2, 3, 128, 104, 64), (0, 3, 256, 40, 64), (4, 3, 256, 72, 64), (0, 3, 512, 24, 64), (2, 3, 1024, 40, 64)])
def test_small_grids_of_any_magnitude(algo, S, DY, K, N, scale, algo_1d):
    print("small grid range", algo, S, DY, K, N, scale, flush=True)
    algo_1d(algo)
    W = _complex(np.random.default_rng(S), N, K) / np.float32(np.sqrt(K))
    run = lambda x, W: tf.layer_1d(x, _dev(W), alpha=0.5 - 0.75j)
    # one product and two transforms in fp32, as bounded in test_gpu_operand_range.py
    tol = 2.0 * (2 * K) ** 0.5 * 2.0 ** -24 + 2 * 16 ** 0.5 * 2.0 ** -24
    _layer_check(run, lambda x, W: oracle.layer_1d(x, W, 0.5 - 0.75j), _x(S, DY, K), W, scale, tol, N)


@pytest.mark.parametrize("DY", [128, 256, 512, 1024])
@pytest.mark.parametrize("S,K,attach", [(20, 64, False), (100, 128, False), (20, 64, True), (300, 40, False)])
def test_y_in_the_place_of_x(S, K, attach, DY):
    """64 output channels: one block per signal set, whatever the size would choose (tiles of 16 or 32, the K split, a cluster):
    nothing of x is overwritten before it is read"""
    N = 64
    print("small grid in place", S, K, attach, DY, flush=True)
    x, W = _x(S, DY, K), _complex(np.random.default_rng(S), N, K) / np.float32(np.sqrt(K))
    ref = oracle.layer_1d(x.cpu().numpy(), W, 1.0)
    buffer = tf.ExchangeBuffer() if attach else None
    try:
        for _ in range(3):
            y = torch.zeros((max(K, N), S, DY), dtype=torch.complex64, device="cuda")
            y[:K] = x
            tf.layer_1d(y[:K], _dev(W), y=y[:N])
            assert rel_l2(y[:N].cpu().numpy(), ref) < _bound(K, 2)
    finally:
        if buffer is not None:
            buffer.close()


@pytest.mark.parametrize("DY", [128, 256, 512, 1024])
def test_halves_of_one_signal_in_place(DY):
    """one signal, 64 output channels: C over x and y over A, read by one block before it writes"""
    N = K = 64
    print("halves in place", DY, flush=True)
    x, W = _x(1, DY, K), _complex(np.random.default_rng(DY), N, K) / np.float32(np.sqrt(K))
    spectra = oracle.fft_trunc_contig(x.cpu().numpy()).reshape(K, 64)
    first = oracle.cgemm(spectra, W, 1.0)
    second = oracle.ifft_pad_contig(oracle.cgemm(first.astype(np.complex64), W, 1.0).reshape(N, 1, 64), DY)
    for _ in range(3):
        buf = x.clone()
        C = buf.view(-1)[:N * 64].view(N, 64)
        tf.fused_fft_cgemm(64, N, K, buf, _dev(W), C)
        assert rel_l2(C.cpu().numpy(), first) < _bound(K, 1)
        buf = torch.zeros((N, 1, DY), dtype=torch.complex64, device="cuda")
        A = buf.view(-1)[:K * 64].view(K, 64)
        A.copy_(torch.from_numpy(first.astype(np.complex64)))
        tf.fused_cgemm_ifft(64, N, K, A, _dev(W), buf)
        assert rel_l2(buf.cpu().numpy(), second) < _bound(K, 1)
