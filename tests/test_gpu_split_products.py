"""fp32 products from three bf16 parts per operand on the matrix cores (csrc/bf16_split.h): the mode GEMM at the edges of its
tiles, steps and runs, against the oracle, and the exactness of the split itself."""
import numpy as np
import pytest
import torch

import oracle
import turbofno_amd as tf
from conftest import max_rel, rel_l2

pytestmark = pytest.mark.gpu


def _complex(rng, *shape):
    return (rng.uniform(-1, 1, shape) + 1j * rng.uniform(-1, 1, shape)).astype(np.complex64)


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


# fp32 sums of 2 K products each: (2 K)^0.5 roundings of 2^-24 each as a random walk, doubled; and in any case less than half of
# what the loss of one of the six partial products costs (l h', h l' or m m': 2.2e-6 to 2.5e-6 of the result for uniform operands at
# every K, from the sums in 64 bits). Measured: 1.5e-7 at K = 64, 2.7e-7 at K = 128 with two transforms.
def _bound(K, transforms=0):
    return min(2.0 * (2 * K) ** 0.5 * 2.0 ** -24 + transforms * 16 ** 0.5 * 2.0 ** -24, 1e-6)      # a transform: eight real additions in a row


@pytest.mark.parametrize("M,K,N,beta", [
    (64, 24, 64, 0.0),               # half a block of columns, a step of which a quarter is beyond K
    (192, 32, 64, 0.0),              # one full step, the second block half filled
    (128, 40, 128, 0.5 - 1j),        # two steps, the last with one quarter wavefront of channels; C read and written
    (320, 96, 192, 0.0),             # three n tiles
    (64, 192, 64, 0.0),              # the largest tile that stays in LDS
    (64, 200, 64, 0.0),              # one step more: the tile is rebuilt, the last build covers one step
    (576, 1000, 64, 1j),             # six builds per column block, a block with idle waves
    (65536 + 64, 72, 64, 0.0),       # more than one block of 256 columns per CU, a partly filled last one
    (524288 + 64, 72, 128, 0.0),     # 128-channel tiles, persistent walk, a partly filled last block
    (4096, 64, 64, 0.0),             # tiles of 16 output channels
    (8192, 200, 128, -1j),           # tiles of 32, the tile rebuilt, C read and written
    (16384, 40, 128, 2.0),           # tiles of 64 in blocks of 128 columns, C read and written
    (32768 + 64, 72, 128, 0.5),      # blocks of 256 columns, the same
    (262144 + 64, 24, 128, 1 + 1j),  # tiles of 128, the same: C is read in two parts
    (262144 - 64, 32, 128, 0.0),     # N = 128 with 32 channels or fewer on a large grid
])
def test_cgemm_edges(M, K, N, beta):
    print("split cgemm", M, K, N, beta, flush=True)
    rng = np.random.default_rng(M + K + N)
    gen = torch.Generator(device="cuda").manual_seed(M + K)
    A = torch.view_as_complex(torch.rand((K, M, 2), device="cuda", generator=gen) * 2 - 1)
    W = _complex(rng, N, K) / np.float32(np.sqrt(K))
    C0 = torch.full((N, M), float("nan"), dtype=torch.complex64, device="cuda") if beta == 0.0 else \
        torch.view_as_complex(torch.rand((N, M, 2), device="cuda", generator=gen) * 2 - 1)
    C = C0.clone()
    tf.cgemm(M, N, K, A, _dev(W), C, 0.5 + 1j, beta)
    torch.cuda.synchronize()
    assert not bool(torch.isnan(torch.view_as_real(C)).any()), "columns of C left unwritten"
    picks = sorted(set(range(0, min(M, 300))) | set(range(max(0, M - 300), M)) | set(range(M // 2, min(M, M // 2 + 32))))
    idx = torch.tensor(picks, device="cuda")
    ref = oracle.cgemm(A.index_select(1, idx).cpu().numpy(), W, 0.5 + 1j)
    if beta != 0.0:
        ref = ref + beta * C0.index_select(1, idx).cpu().numpy().astype(np.complex128)
    err = rel_l2(C.index_select(1, idx).cpu().numpy(), ref)
    assert err < _bound(K), (err, _bound(K))


@pytest.mark.parametrize("K", [24, 64])
def test_split_is_exact(K):
    """weights 1, i, -1 and 2^-20 on one channel each: nothing is rounded, so the product is the input bit for bit. Inputs over
    the range in which all three parts are normal numbers, with full 24-bit significands."""
    print("split exact", K, flush=True)
    rng = np.random.default_rng(K)
    M, N = 256, 64
    mant = rng.integers(2 ** 23, 2 ** 24, (K, M, 2)).astype(np.float64) * rng.choice([-1.0, 1.0], (K, M, 2))
    A = np.ldexp(mant, rng.integers(-80, 100, (K, M, 2))).astype(np.float32).view(np.complex64)[..., 0]
    W = np.zeros((N, K), np.complex64)
    factor = np.array([1, 1j, -1, 2.0 ** -20], np.complex64)
    for n in range(N):
        W[n, (5 * n) % K] = factor[n % 4]
    C = torch.empty((N, M), dtype=torch.complex64, device="cuda")
    tf.cgemm(M, N, K, _dev(A), _dev(W), C, 1.0, 0.0)
    got = C.cpu().numpy()
    for n in range(N):
        f, a = factor[n % 4], A[(5 * n) % K]
        want = np.empty_like(a)
        want.real, want.imag = (-a.imag, a.real) if f == 1j else (a.real * f.real, a.imag * f.real)
        assert np.array_equal(got[n].real, want.real) and np.array_equal(got[n].imag, want.imag), n


def _significands(rng, *shape):
    """values with all 24 bits in use, over 40 binades"""
    mant = rng.integers(2 ** 23, 2 ** 24, shape).astype(np.float64) * rng.choice([-1.0, 1.0], shape)
    return np.ldexp(mant, rng.integers(-43, -3, shape)).astype(np.float32)


# one product: 2^-24 for the three partial products that are left out, one spacing (2^-23) for the last sum - a matrix instruction adds
# its products and the accumulator without rounding to nearest: 1.27e-7 was seen, above the 2 x 2^-24 of a nearest sum - and 2^-31 for
# each of the small ones before it; the loss of l h' or of m m' costs up to 2^-17 and 2^-16
SINGLE = 3.1 * 2.0 ** -24


def _single_weights(rng, N, K):
    """per output channel one weight, real or imaginary in turn; its channel"""
    r, k = _significands(rng, N), (5 * np.arange(N) + 3) % K
    W = np.zeros((N, K), np.complex64)
    W[np.arange(N), k] = np.where(np.arange(N) % 2 == 0, r, 1j * r)
    return W, k


@pytest.mark.parametrize("M,K,N", [(64, 24, 64), (128, 200, 64), (8192, 40, 128), (16384, 64, 128), (32768 + 64, 72, 128), (524288, 40, 128)])
def test_single_products_of_the_mode_gemm(M, K, N):
    print("single products cgemm", M, K, N, flush=True)
    rng = np.random.default_rng(M + K)
    W, k = _single_weights(rng, N, K)
    head = _significands(rng, K, 64).astype(np.complex64)
    A = torch.zeros((K, M), dtype=torch.complex64, device="cuda")
    A[:, :64] = _dev(head)
    A[:, M - 64:] = _dev(head)
    C = torch.full((N, M), float("nan"), dtype=torch.complex64, device="cuda")
    tf.cgemm(M, N, K, A, _dev(W), C, 1.0, 0.0)
    want = W[np.arange(N), k].astype(np.complex128)[:, None] * head.astype(np.complex128)[k]
    for got in (C[:, :64], C[:, M - 64:]):
        assert np.max(np.abs(got.cpu().numpy() - want) / np.abs(want)) < SINGLE
    assert not bool(C[:, 64:M - 64].any())


@pytest.mark.parametrize("algo,S,DY,K,N", [
    (6, 3, 256, 64, 64), (6, 5, 256, 136, 128), (6, 9, 256, 256, 64),       # the channels split over the waves
    (3, 5, 128, 40, 64), (3, 5, 256, 40, 64), (5, 5, 256, 40, 64), (3, 5, 512, 40, 64), (3, 5, 1024, 40, 64),
    (8, 5, 128, 40, 128), (8, 5, 256, 40, 128), (8, 5, 512, 40, 128), (8, 5, 1024, 40, 128),
])
def test_single_products_of_the_1d_kernels(algo, S, DY, K, N, algo_1d):
    """constant signals: the spectrum is DY times the value at mode 0 and zero elsewhere, without a rounding, and back; so every
    sample of an output signal is DY times one product"""
    print("single products 1d", algo, S, DY, K, N, flush=True)
    algo_1d(algo)
    assert tf.query_1d_kernel(DY, S, N, K) == algo
    rng = np.random.default_rng(S + DY + K)
    W, k = _single_weights(rng, N, K)
    v = _significands(rng, K, S).astype(np.complex64)
    x = np.repeat(v[:, :, None], DY, axis=2)
    want = W[np.arange(N), k].astype(np.complex128)[:, None] * v.astype(np.complex128)[k] * DY
    y = tf.layer_1d(_dev(x), _dev(W)).cpu().numpy()
    assert np.max(np.abs(y - want[:, :, None]) / np.abs(want)[:, :, None]) < SINGLE
    # the halves: spectra of the constant signals, backward transforms of a product with mode 0 alone
    C = torch.empty((N, S, 64), dtype=torch.complex64, device="cuda")
    tf.fused_fft_cgemm(64 * S, N, K, _dev(x), _dev(W), C, 1.0, 0.0)
    C = C.cpu().numpy()
    assert np.max(np.abs(C[:, :, 0] - want) / np.abs(want)) < SINGLE and not C[:, :, 1:].any()
    A = np.zeros((K, S, 64), np.complex64)
    A[:, :, 0] = v
    y = torch.empty((N, S, DY), dtype=torch.complex64, device="cuda")
    tf.fused_cgemm_ifft(64 * S, N, K, _dev(A), _dev(W), y, 1.0)
    assert np.max(np.abs(y.cpu().numpy() * DY - want[:, :, None]) / np.abs(want)[:, :, None]) < SINGLE


@pytest.mark.parametrize("S,K,N", [(1, 64, 64), (40, 72, 128), (64, 104, 64), (7, 136, 192), (32, 256, 128)])
def test_small_grids_with_many_channels(S, K, N, algo_1d):
    """the kernel that splits the channels over its waves, under the bound for split products"""
    print("split small grids", S, K, N, flush=True)
    algo_1d(6)
    assert tf.query_1d_kernel(256, S, N, K) == 6
    rng = np.random.default_rng(S + K)
    x, W = _complex(rng, K, S, 256), _complex(rng, N, K) / np.float32(np.sqrt(K))
    y = tf.layer_1d(_dev(x), _dev(W), alpha=0.5 - 0.75j)
    assert rel_l2(y.cpu().numpy(), oracle.layer_1d(x, W, 0.5 - 0.75j)) < _bound(K, 2)


@pytest.mark.parametrize("bs,DX,DY,K,N", [(2, 512, 128, 8, 64), (1, 512, 256, 40, 64), (1, 1024, 128, 24, 128), (1, 1024, 128, 104, 64),
                                          (1, 512, 128, 64, 64), (1, 512, 128, 200, 64), (1, 512, 128, 16, 64), (2, 512, 128, 24, 128), (1, 1024, 128, 40, 64),
                                          (5, 512, 128, 72, 128)])
def test_weights_with_a_period(bs, DX, DY, K, N):
    """whole images in 2 / 4 interleaved parts: the contraction runs over the parts with the weights of their channel, as one
    run over all parts (K = 8, 24, 40) or as one run per part (K = 64, 104; K = 200 with a tile that is rebuilt); K = 16, 40 and 24, 72: a run
    whose last step is full and short where that of a part is not"""
    print("split period", bs, DX, DY, K, N, flush=True)
    rng = np.random.default_rng(DX + K)
    x, W = _complex(rng, K, bs, DX, DY), _complex(rng, N, K) / np.float32(np.sqrt(K))
    y = tf.layer_2d(_dev(x), _dev(W), algo=2, alpha=1 - 1j)
    torch.cuda.synchronize()
    ref = oracle.layer_2d(x, W, 1 - 1j)
    assert rel_l2(y.cpu().numpy(), ref) < 1e-6 and max_rel(y.cpu().numpy(), ref) < 1e-5


@pytest.mark.parametrize("M", [64, 4096, 65536 + 64])
def test_mode_gemm_in_place(M):
    """64 output channels over the 64 input channels"""
    print("split cgemm in place", M, flush=True)
    rng = np.random.default_rng(M)
    A, W = _complex(rng, 64, M), _complex(rng, 64, 64)
    C = _dev(A)
    for _ in range(3):
        C.copy_(torch.from_numpy(A))
        tf.cgemm(M, 64, 64, C, _dev(W), C, 1.0, 0.0)
        assert rel_l2(C.cpu().numpy(), oracle.cgemm(A, W, 1.0)) < _bound(64)


# of the shapes below, those with 128 output channels per block
WIDE = {(512, 256, 128, 128), (912, 256, 72, 128), (513, 128, 104, 128), (1100, 128, 96, 256), (520, 512, 104, 128), (193, 1024, 8, 128),
        (256, 1024, 72, 128), (1024, 256, 72, 128)}


@pytest.mark.parametrize("S,DY,K,N", [
    (224, 256, 8, 64),               # half a round: two of four waves without a transform
    (300, 256, 40, 192),             # a short last round, three blocks of 64 channels per signal set
    (900, 256, 24, 64),              # four blocks per CU
    (130, 256, 16, 256),             # a tail of two signal sets behind the groups of eight
    (512, 256, 128, 128),            # blocks of 128 channels
    (912, 256, 72, 128),             # the same with a short last round
    (200, 128, 40, 64),              # DY = 128: rounds of 32 channels, the last with eight
    (257, 128, 24, 192),             # one round of 24
    (260, 128, 16, 64),              # half a round: the second step of the product is skipped
    (513, 128, 104, 128),            # blocks of 128 channels, the last round with eight
    (560, 128, 56, 256),             # 24 in the last round, four blocks of 64 per signal set
    (1100, 128, 96, 256),            # blocks of 128 channels, two per signal set
    (260, 512, 40, 64),              # DY = 512: two passes per round, the last round with one
    (140, 512, 32, 128),             # blocks of 64 channels with N = 128
    (520, 512, 104, 128),            # blocks of 128 channels
    (258, 1024, 40, 64),             # DY = 1024: four passes per round, the last round with two
    (193, 1024, 8, 128),             # blocks of 128 channels, half a round
    (256, 1024, 72, 128),            # the same with a short last round
    (512, 256, 24, 64),              # 1 and 2 MiB between channels: the waves of a block take every fourth output channel
    (1024, 256, 72, 128),            # the same with blocks of 128 channels
    (512, 512, 40, 192),
    (512, 1024, 72, 64),             # 4 MiB: neighbouring channels again
])
def test_fused_1d_edges(S, DY, K, N):
    """the fused 1D kernel with split products, chosen by size: every row of y written (y starts as NaN), the first, last and
    some inner signal sets against the oracle"""
    print("split fused 1d", S, DY, K, N, flush=True)
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert tf.query_1d_kernel(DY, S, N, K, compute_units=0) in (3, 5, 8)
        assert tf.query_1d_tile(DY, S, N, K, compute_units=0) == (128 if (S, DY, K, N) in WIDE else 64)
    gen = torch.Generator(device="cuda").manual_seed(S + DY + K)
    x = torch.view_as_complex(torch.rand((K, S, DY, 2), device="cuda", generator=gen) * 2 - 1)
    W = _complex(np.random.default_rng(S), N, K) / np.float32(np.sqrt(K))
    y = torch.full((N, S, DY), float("nan"), dtype=torch.complex64, device="cuda")
    tf.layer_1d(x, _dev(W), y=y, alpha=0.5 - 0.75j)
    torch.cuda.synchronize()
    assert not bool(torch.isnan(torch.view_as_real(y)).any()), "rows of y left unwritten"
    idx = torch.tensor(sorted({0, 1, 7, 8, S // 2, S - 9, S - 2, S - 1}), device="cuda")
    ref = oracle.layer_1d(x.index_select(1, idx).cpu().numpy(), W, 0.5 - 0.75j)
    err = rel_l2(y.index_select(1, idx).cpu().numpy(), ref)
    assert err < _bound(K, 2), err


@pytest.mark.parametrize("S,DY,K,N", [
    (1, 128, 8, 128), (11, 128, 72, 256), (2048, 128, 40, 256),      # S = 2048, 4096: XCD j walks the j-th eighth of the signal sets
    (3, 256, 72, 256), (2048, 256, 32, 256), (13, 512, 24, 256), (1024, 512, 40, 128), (2, 1024, 8, 128), (130, 1024, 40, 256),
])
def test_blocks_of_128_output_channels(S, DY, K, N, algo_1d):
    """forced by the selector at sizes where the rule takes other blocks: one and two blocks per signal set, both block orders"""
    print("split 128 outputs", S, DY, K, N, flush=True)
    algo_1d(8)
    assert tf.query_1d_kernel(DY, S, N, K) == 8 and tf.query_1d_tile(DY, S, N, K) == 128
    gen = torch.Generator(device="cuda").manual_seed(S + DY + K)
    x = torch.view_as_complex(torch.rand((K, S, DY, 2), device="cuda", generator=gen) * 2 - 1)
    W = _complex(np.random.default_rng(S), N, K) / np.float32(np.sqrt(K))
    y = torch.full((N, S, DY), float("nan"), dtype=torch.complex64, device="cuda")
    tf.layer_1d(x, _dev(W), y=y, alpha=0.5 - 0.75j)
    torch.cuda.synchronize()
    assert not bool(torch.isnan(torch.view_as_real(y)).any()), "rows of y left unwritten"
    e = S // 8
    idx = torch.tensor(sorted({0, S // 2, S - 1} | {p for p in (7, 8, e - 1, e, 7 * e) if 0 <= p < S}), device="cuda")
    ref = oracle.layer_1d(x.index_select(1, idx).cpu().numpy(), W, 0.5 - 0.75j)
    err = rel_l2(y.index_select(1, idx).cpu().numpy(), ref)
    assert err < _bound(K, 2), err


@pytest.mark.parametrize("algo", [1, 3])
@pytest.mark.parametrize("bs,DX,DY,K,N", [(1, 128, 256, 16, 128), (2, 256, 128, 40, 256), (1, 512, 256, 24, 128), (1, 256, 512, 40, 128),
                                          (1, 1024, 512, 8, 128), (1, 512, 1024, 8, 128)])
def test_blocks_of_128_output_channels_as_middle_stage(bs, DX, DY, K, N, algo, algo_1d):
    """the same as the middle stage of a 2D layer of three kernels: plain stores"""
    print("split 128 outputs middle", bs, DX, DY, K, N, algo, flush=True)
    algo_1d(8)
    rng = np.random.default_rng(DX + DY)
    x, W = _complex(rng, K, bs, DX, DY), _complex(rng, N, K) / np.float32(np.sqrt(K))
    y = tf.layer_2d(_dev(x), _dev(W), algo=algo, alpha=1 - 1j)
    torch.cuda.synchronize()
    ref = oracle.layer_2d(x, W, 1 - 1j)
    assert rel_l2(y.cpu().numpy(), ref) < 1e-6 and max_rel(y.cpu().numpy(), ref) < 1e-5


@pytest.mark.parametrize("S,DY,K,N", [
    (1, 128, 8, 64), (9, 128, 40, 192), (400, 128, 56, 128),        # rounds of 32 channels: one of eight, a last one of eight, of 24
    (1, 256, 8, 64), (9, 256, 40, 192), (400, 256, 72, 128),        # S = 400: blocks of 128 output channels
    (160, 128, 56, 64),                                              # first half with a short round, less than one block per CU
    (3, 512, 24, 64), (400, 512, 40, 128), (2, 1024, 8, 64), (390, 1024, 24, 128),
    (5, 512, 8, 192), (900, 1024, 8, 64), (3, 1024, 16, 128),       # few channels; the second: first half by the SIMT kernel
    (512, 256, 40, 64), (256, 512, 40, 128), (128, 1024, 24, 64),   # 1 MiB between channels: the waves of a block take every fourth one
])
@pytest.mark.parametrize("beta", [0.0, -1 + 1j])
def test_halves_of_the_layer(S, DY, K, N, beta):
    """forward transforms with the product (every value of C written, or added to with beta), product with backward transforms"""
    print("split halves", S, DY, K, N, beta, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(S + DY + K)
    rng = np.random.default_rng(S + K)
    x = torch.view_as_complex(torch.rand((K, S, DY, 2), device="cuda", generator=gen) * 2 - 1)
    W, W2 = _complex(rng, N, K) / np.float32(np.sqrt(K)), _complex(rng, N, N) / np.float32(np.sqrt(N))
    C0 = torch.full((N, S, 64), float("nan"), dtype=torch.complex64, device="cuda") if beta == 0.0 else \
        torch.view_as_complex(torch.rand((N, S, 64, 2), device="cuda", generator=gen) * 2 - 1)
    C = C0.clone()
    tf.fused_fft_cgemm(64 * S, N, K, x, _dev(W), C, 0.5 - 0.75j, beta)
    y = torch.full((N, S, DY), float("nan"), dtype=torch.complex64, device="cuda")
    tf.fused_cgemm_ifft(64 * S, N, N, C, _dev(W2), y, 1 - 1j)
    torch.cuda.synchronize()
    assert not bool(torch.isnan(torch.view_as_real(C)).any()), "values of C left unwritten"
    assert not bool(torch.isnan(torch.view_as_real(y)).any()), "rows of y left unwritten"
    idx = torch.tensor(sorted({0, S // 2, max(0, S - 9), S - 1}), device="cuda")
    pick = lambda a: a.index_select(1, idx).cpu().numpy()
    ref = oracle.cgemm(oracle.fft_trunc_contig(pick(x)).reshape(K, -1), W, 0.5 - 0.75j).reshape(N, -1, 64)
    if beta != 0.0:
        ref = ref + beta * pick(C0).astype(np.complex128)
    assert rel_l2(pick(C), ref) < _bound(K, 1)
    ref = oracle.ifft_pad_contig(oracle.cgemm(pick(C).reshape(N, -1), W2, 1 - 1j).reshape(N, -1, 64), DY)
    assert rel_l2(pick(y), ref) < _bound(N, 1)


@pytest.mark.parametrize("S,DY,N", [
    (300, 512, 64), (900, 1024, 64),     # both halves by the SIMT kernel (first half at 1024: three to eight blocks per CU)
    (300, 1024, 64),                     # the second
    (240, 512, 64),                      # the second, between seven eighths of a block and a block per CU
    (150, 512, 192),                     # both, three blocks per signal set
])
@pytest.mark.parametrize("beta", [0.0, -1 + 1j])
def test_halves_with_eight_channels_on_larger_grids(S, DY, N, beta):
    """the SIMT kernel, which sums in fp32 without splits: every value of C and y written, the halves apart from each other"""
    K = 8
    print("SIMT halves", S, DY, N, beta, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(S + DY)
    rng = np.random.default_rng(S + N)
    x = torch.view_as_complex(torch.rand((K, S, DY, 2), device="cuda", generator=gen) * 2 - 1)
    A = torch.view_as_complex(torch.rand((K, S, 64, 2), device="cuda", generator=gen) * 2 - 1)
    W = _complex(rng, N, K) / np.float32(np.sqrt(K))
    C0 = torch.full((N, S, 64), float("nan"), dtype=torch.complex64, device="cuda") if beta == 0.0 else \
        torch.view_as_complex(torch.rand((N, S, 64, 2), device="cuda", generator=gen) * 2 - 1)
    C, y = C0.clone(), torch.full((N, S, DY), float("nan"), dtype=torch.complex64, device="cuda")
    tf.fused_fft_cgemm(64 * S, N, K, x, _dev(W), C, 0.5 - 0.75j, beta)
    tf.fused_cgemm_ifft(64 * S, N, K, A, _dev(W), y, 1 - 1j)
    torch.cuda.synchronize()
    assert not bool(torch.isnan(torch.view_as_real(C)).any()), "values of C left unwritten"
    assert not bool(torch.isnan(torch.view_as_real(y)).any()), "rows of y left unwritten"
    idx = torch.tensor(sorted({0, 7, S // 2, S - 9, S - 1}), device="cuda")
    pick = lambda a: a.index_select(1, idx).cpu().numpy()
    ref = oracle.cgemm(oracle.fft_trunc_contig(pick(x)).reshape(K, -1), W, 0.5 - 0.75j).reshape(N, -1, 64)
    if beta != 0.0:
        ref = ref + beta * pick(C0).astype(np.complex128)
    assert rel_l2(pick(C), ref) < _bound(K, 1)
    ref = oracle.ifft_pad_contig(oracle.cgemm(pick(A).reshape(K, -1), W, 1 - 1j).reshape(N, -1, 64), DY)
    assert rel_l2(pick(y), ref) < _bound(K, 1)
