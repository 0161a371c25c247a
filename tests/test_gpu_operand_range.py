"""Products of operands outside the range of the three-way bf16 split (csrc/bf16_split.h): magnitudes down to the smallest normal
float, up to the largest one, infinities and NaN give what fp32 arithmetic gives."""
import numpy as np
import pytest
import torch

import oracle
import turbofno_amd as tf

pytestmark = pytest.mark.gpu


def _complex(rng, *shape):
    return (rng.uniform(-1, 1, shape) + 1j * rng.uniform(-1, 1, shape)).astype(np.complex64)


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


# fp32 sums of 2 K products each: (2 K)^0.5 roundings of 2^-24 as a random walk, doubled (single rows and columns: not the cap that the
# tests of whole results have)
def _bound(K):
    return 2.0 * (2 * K) ** 0.5 * 2.0 ** -24


def _worst(got, ref, axis):
    """largest relative 2-norm error of a row (axis 1) or column (axis 0)"""
    return float(np.max(np.linalg.norm(got - ref, axis=axis) / np.linalg.norm(ref, axis=axis)))


CGEMM = [
    (64, 24, 64, 0.0),               # tiles of 16 output channels
    (128, 40, 128, 0.5 - 1j),        # C read and written
    (64, 200, 64, 0.0),              # weights rebuilt in LDS as the contraction proceeds
    (8192, 64, 128, 0.0),            # tiles of 32
    (65536 + 64, 72, 64, 0.0),       # tiles of 64 in blocks of 128 columns that walk several of them
    (32768 + 64, 72, 128, 0.5),      # blocks of 256 columns
    (524288 + 64, 72, 128, 0.0),     # tiles of 128 output channels
]


def _cgemm(A, W, beta, C0):
    K, M = A.shape
    N = W.shape[0]
    C = C0.clone()
    tf.cgemm(M, N, K, A, _dev(W), C, 1.0, beta)
    torch.cuda.synchronize()
    return C


@pytest.mark.parametrize("scale", [1e-33, 1e-35, 1e-37, 1e37])
@pytest.mark.parametrize("M,K,N,beta", CGEMM)
def test_cgemm_operands_of_any_magnitude(M, K, N, beta, scale):
    """strips of columns of A, then every third row of W, at the given magnitude among others near one"""
    print("cgemm range", M, K, N, beta, scale, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(M + K)
    rng = np.random.default_rng(M + K)
    A = torch.view_as_complex(torch.rand((K, M, 2), device="cuda", generator=gen) * 2 - 1)
    W = _complex(rng, N, K) / np.float32(np.sqrt(K))
    C0 = torch.view_as_complex(torch.rand((N, M, 2), device="cuda", generator=gen) * 2 - 1) * np.float32(scale)
    picks = sorted(set(range(0, 64)) | set(range(M - 64, M)) | set(range(M // 2 - 16, M // 2 + 16)))
    idx = torch.tensor(picks, device="cuda")
    small = idx[(idx % 32) < 20]
    As = A.clone()
    As[:, small] *= scale
    Cs = _cgemm(As, W, beta, C0)
    ref = oracle.cgemm(As.index_select(1, idx).cpu().numpy(), W, 1.0) + beta * C0.index_select(1, idx).cpu().numpy().astype(np.complex128)
    assert _worst(Cs.index_select(1, idx).cpu().numpy(), ref, 0) < _bound(K)
    Ws = W.copy()
    Ws[::3] *= np.float32(scale)
    if beta != 0.0:
        C0[1::3] /= np.float32(scale)
        C0[2::3] /= np.float32(scale)
    Cs = _cgemm(A, Ws, beta, C0)
    ref = oracle.cgemm(A.index_select(1, idx).cpu().numpy(), Ws, 1.0) + beta * C0.index_select(1, idx).cpu().numpy().astype(np.complex128)
    assert _worst(Cs.index_select(1, idx).cpu().numpy(), ref, 1) < _bound(K)


@pytest.mark.parametrize("M,K,N,beta", CGEMM[:3])
def test_cgemm_magnitudes_mixed_in_one_sum(M, K, N, beta):
    """small values of A that only small weights, or only weights near one, meet"""
    print("cgemm mixed range", M, K, N, flush=True)
    rng = np.random.default_rng(M + K)
    A, W = _complex(rng, K, M), _complex(rng, N, K)
    A[K // 2:] *= np.float32(1e-37)
    W[:N // 2, :K // 2] = 0.0                # rows whose result is at 1e-37
    W[N // 2:, K // 2:] *= np.float32(1e30)
    W[N // 2:, :K // 2] *= np.float32(1e-10)
    C = _cgemm(_dev(A), W, 0.0, torch.empty((N, M), dtype=torch.complex64, device="cuda")).cpu().numpy()
    assert _worst(C, oracle.cgemm(A, W, 1.0), 1) < _bound(K)


def _fp32_classes(A, W):
    """(is infinite, is NaN) of the real and imaginary parts of W A in real arithmetic"""
    with np.errstate(all="ignore"):
        A, W = A.astype(np.complex128), W.astype(np.complex128)
        re = np.zeros((W.shape[0], A.shape[1]))
        im = np.zeros_like(re)
        for k in range(A.shape[0]):
            w, a = W[:, k:k + 1], A[k:k + 1]
            re = re + w.real * a.real - w.imag * a.imag
            im = im + w.real * a.imag + w.imag * a.real
    v = np.stack([re, im])
    return np.isinf(v), np.isnan(v), v


@pytest.mark.parametrize("value", [complex(np.inf, 0), complex(0, -np.inf), complex(np.nan, 1), complex(3.4e38, 0), complex(0, -3.4028234e38)])
@pytest.mark.parametrize("M,K,N,beta", [(64, 24, 64, 0.0), (128, 40, 128, 0.0), (64, 200, 64, 0.0)])
def test_cgemm_infinities_and_the_largest_floats(M, K, N, beta, value):
    """one such value in A, then in W: the same infinities, NaN and finite results as real fp32 arithmetic"""
    print("cgemm infinities", M, K, N, value, flush=True)
    rng = np.random.default_rng(M + K)
    for where in "AW":
        A, W = _complex(rng, K, M) * np.float32(0.01), _complex(rng, N, K) * np.float32(0.01)
        (A if where == "A" else W)[5, 17] = value
        C = torch.empty((N, M), dtype=torch.complex64, device="cuda")
        tf.cgemm(M, N, K, _dev(A), _dev(W), C, 1.0, 0.0)
        got = C.cpu().numpy()
        got = np.stack([got.real, got.imag])
        # alpha = 1 + 0i is multiplied into W first: an infinite weight becomes inf * 1 - x * 0 and x * 1 + inf * 0 = NaN
        if where == "W" and not np.isfinite(value):
            W[5, 17] = complex(value.real * 1.0 - value.imag * 0.0, value.real * 0.0 + value.imag * 1.0)
        inf, nan, ref = _fp32_classes(A, W)
        assert np.array_equal(np.isnan(got), nan) and np.array_equal(np.isinf(got), inf), where
        assert np.array_equal(np.sign(got[inf]), np.sign(ref[inf]))
        fine = ~(inf | nan)
        scale = np.maximum(np.abs(ref[fine]), 0.01 * 0.01)
        assert np.max(np.abs(got[fine] - ref[fine]) / scale) < 2 * K * 2.0 ** -24 + 1e-5


LAYERS = [                           # S, DY, K, N: the fused 1D kernel with 64 and 128 output channels per block
    (260, 128, 40, 64), (513, 128, 104, 128),
    (300, 256, 40, 64), (900, 256, 24, 64), (512, 256, 128, 128),
    (260, 512, 40, 64), (520, 512, 104, 128),
    (258, 1024, 40, 64), (256, 1024, 72, 128),
    (512, 256, 40, 64), (512, 512, 40, 64),                          # 1 and 2 MiB between channels: waves of every fourth channel
]
SMALL_GRIDS = [(3, 64, 64), (5, 136, 128), (9, 128, 192)]     # S, K, N at DY = 256: the channels split over the waves of a block
HALVES = [(9, 128, 40, 64), (513, 128, 40, 128), (9, 256, 72, 64), (400, 256, 40, 128), (9, 512, 40, 64), (400, 512, 40, 128),
          (9, 1024, 40, 64), (390, 1024, 24, 128), (256, 512, 24, 64), (128, 1024, 8, 128),
          (300, 512, 8, 64)]                     # the SIMT kernel
_TRANSFORMS = 2 * 16 ** 0.5 * 2.0 ** -24       # two transforms of eight real additions in a row per value


def _layer_check(run, reference, x, W, scale, tol, channels_out):
    """run(x, W) with some signal sets, then with some rows of W at `scale`: relative error of every signal set / output channel"""
    S = x.shape[1]
    sets = sorted({0, S // 2, S - 1})
    idx = torch.tensor(sets, device="cuda")
    xs = x.clone()
    xs[:, idx[1:]] *= scale
    y = run(xs, W)
    assert not bool(torch.isnan(torch.view_as_real(y)).any())
    pick = lambda a: a.index_select(1, idx).cpu().numpy()
    ref = reference(pick(xs), W)
    for i in range(len(sets)):
        err = np.linalg.norm(pick(y)[:, i] - ref[:, i]) / np.linalg.norm(ref[:, i])
        assert err < tol, ("signal set", sets[i], err)
    Ws = W.copy()
    Ws[1::3] *= np.float32(scale)
    y = pick(run(x, Ws))
    ref = reference(pick(x), Ws)
    for n in range(channels_out):
        err = np.linalg.norm(y[n] - ref[n]) / np.linalg.norm(ref[n])
        assert err < tol, ("output channel", n, err)


def _x(S, L, K):
    gen = torch.Generator(device="cuda").manual_seed(S + L + K)
    return torch.view_as_complex(torch.rand((K, S, L, 2), device="cuda", generator=gen) * 2 - 1)


@pytest.mark.parametrize("scale", [1e-35, 1e-37, 1e20])
@pytest.mark.parametrize("S,DY,K,N", LAYERS)
def test_layer_1d_of_any_magnitude(S, DY, K, N, scale):
    print("layer range", S, DY, K, N, scale, flush=True)
    W = _complex(np.random.default_rng(S), N, K) / np.float32(np.sqrt(K))
    run = lambda x, W: tf.layer_1d(x, _dev(W), alpha=0.5 - 0.75j)
    _layer_check(run, lambda x, W: oracle.layer_1d(x, W, 0.5 - 0.75j), _x(S, DY, K), W, scale, _bound(K) + _TRANSFORMS, N)


@pytest.mark.parametrize("scale", [1.0, 1e-35, 1e-37, 1e20])
@pytest.mark.parametrize("S,K,N", SMALL_GRIDS)
def test_small_grids_of_any_magnitude(S, K, N, scale, algo_1d):
    print("small grid range", S, K, N, scale, flush=True)
    algo_1d(6)
    assert tf.query_1d_kernel(256, S, N, K) == 6
    W = _complex(np.random.default_rng(S), N, K) / np.float32(np.sqrt(K))
    run = lambda x, W: tf.layer_1d(x, _dev(W), alpha=0.5 - 0.75j)
    _layer_check(run, lambda x, W: oracle.layer_1d(x, W, 0.5 - 0.75j), _x(S, 256, K), W, scale, _bound(K) + _TRANSFORMS, N)


@pytest.mark.parametrize("scale", [1e-35, 1e-37, 1e20])
@pytest.mark.parametrize("S,DY,K,N", HALVES)
def test_halves_of_the_layer_of_any_magnitude(S, DY, K, N, scale):
    print("halves range", S, DY, K, N, scale, flush=True)
    W = _complex(np.random.default_rng(S), N, K) / np.float32(np.sqrt(K))

    def forward(x, W):
        C = torch.empty((N, S, 64), dtype=torch.complex64, device="cuda")
        tf.fused_fft_cgemm(64 * S, N, K, x, _dev(W), C, 1.0, 0.0)
        return C

    def backward(A, W):
        y = torch.empty((N, S, DY), dtype=torch.complex64, device="cuda")
        tf.fused_cgemm_ifft(64 * S, N, K, A, _dev(W), y, 1.0)
        return y

    product = lambda A, W: oracle.cgemm(A.reshape(K, -1), W, 1.0).reshape(N, -1, 64)
    _layer_check(forward, lambda x, W: product(oracle.fft_trunc_contig(x), W), _x(S, DY, K), W, scale, _bound(K) + _TRANSFORMS, N)
    _layer_check(backward, lambda A, W: oracle.ifft_pad_contig(product(A, W), DY), _x(S, 64, K), W, scale, _bound(K) + _TRANSFORMS, N)


@pytest.mark.parametrize("DY", [128, 256, 512, 1024])
def test_halves_with_the_largest_floats(DY):
    """values within a bf16 rounding of the largest float, whose products and transforms are in range again; infinities reach the
    outputs that depend on them and no others"""
    print("halves largest", DY, flush=True)
    S, K, N = 3, 24, 64
    rng = np.random.default_rng(DY)
    A, W = _complex(rng, K, S, 64), _complex(rng, N, K) * np.float32(1e-4)
    A[5, 1, 9] = 3.4e38 - 3.4028234e38j
    y = torch.empty((N, S, DY), dtype=torch.complex64, device="cuda")
    tf.fused_cgemm_ifft(64 * S, N, K, _dev(A), _dev(W), y, 1.0)
    ref = oracle.ifft_pad_contig(oracle.cgemm(A.reshape(K, -1), W, 1.0).reshape(N, S, 64), DY)
    y = y.cpu().numpy().astype(np.complex128)
    for s in range(S):
        assert np.linalg.norm(y[:, s] - ref[:, s]) / np.linalg.norm(ref[:, s]) < _bound(K) + _TRANSFORMS
    x, W = _complex(rng, K, S, DY) * np.float32(1e-4), _complex(rng, N, K)
    W[11, 7] = 3.4e38 + 1j
    C = torch.empty((N, S, 64), dtype=torch.complex64, device="cuda")
    tf.fused_fft_cgemm(64 * S, N, K, _dev(x), _dev(W), C, 1.0, 0.0)
    ref = oracle.cgemm(oracle.fft_trunc_contig(x).reshape(K, -1), W, 1.0).reshape(N, S, 64)
    C = C.cpu().numpy().astype(np.complex128)
    for n in range(N):
        assert np.linalg.norm(C[n] - ref[n]) / np.linalg.norm(ref[n]) < _bound(K) + _TRANSFORMS
    W[11, 7] = np.inf
    C = torch.empty((N, S, 64), dtype=torch.complex64, device="cuda")
    tf.fused_fft_cgemm(64 * S, N, K, _dev(x), _dev(W), C, 1.0, 0.0)
    bad = ~np.isfinite(C.cpu().numpy())
    assert bad[11].all() and not np.delete(bad, 11, axis=0).any()
