"""Row kernels of the rows-first 2D path with 8, 16 and 32 rows per block (csrc/rows_fft.hip): calls on both sides of each limit, against an fp64
evaluation of the same definition by torch.fft on the GPU."""
import pytest
import torch

import turbofno_amd as tf

pytestmark = pytest.mark.gpu


# rows per CU (256 CUs) of the forward kernel (K bs DX) and of the backward kernel (N bs DX), and the rows per block they run with
@pytest.mark.parametrize("bs,DX,DY,K,N", [
    (1, 128, 256, 8, 64),            # 4, 32: 16 and 16
    (2, 128, 256, 40, 64),           # 40, 64: 32 and 32
    (1, 128, 512, 32, 64),           # 16, 32: 8 and 16
    (1, 512, 512, 32, 64),           # 64, 128: 16 and 32
    (3, 256, 512, 24, 64),           # 72, 192: 32 and 32
    (1, 128, 1024, 8, 128),          # 4, 64: 8 and 8
    (1, 512, 1024, 40, 64),          # 80, 128: 16 and 8
    (1, 1024, 1024, 40, 64),         # 160, 256: 32 and 32
])
def test_rows_first(bs, DX, DY, K, N):
    print("row blocks", bs, DX, DY, K, N, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(DX + DY + K)
    x = torch.view_as_complex(torch.rand((K, bs, DX, DY, 2), device="cuda", generator=gen) * 2 - 1)
    W = torch.view_as_complex(torch.rand((N, K, 2), device="cuda", generator=gen) * 2 - 1)
    y = torch.full((N, bs, DX, DY), float("nan"), dtype=torch.complex64, device="cuda")
    tf.layer_2d(x, W, y=y, algo=tf.ALGO_ROWS_FIRST)
    assert not bool(torch.isnan(torch.view_as_real(y)).any()), "rows of y left unwritten"
    modes = torch.stack([torch.fft.fft2(x[k].to(torch.complex128))[..., :64, :64] for k in range(K)])
    mixed = torch.matmul(W.to(torch.complex128), modes.reshape(K, -1)).reshape(N, bs, 64, 64)
    difference = square = 0.0
    for n in range(N):
        padded = torch.zeros((bs, DX, DY), dtype=torch.complex128, device="cuda")
        padded[:, :64, :64] = mixed[n]
        ref = torch.fft.ifft2(padded) * (DX * DY)
        difference += float(torch.linalg.vector_norm(y[n] - ref) ** 2)
        square += float(torch.linalg.vector_norm(ref) ** 2)
    # a product of 2 K terms and four transforms of at most ten additions in a row, fp32, doubled
    bound = 2.0 * ((2 * K) ** 0.5 + 4 * 10 ** 0.5) * 2.0 ** -24
    assert (difference / square) ** 0.5 < bound, ((difference / square) ** 0.5, bound)
