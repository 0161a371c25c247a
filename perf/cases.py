"""What the speed of this framework is measured on: cases through the public entry points of `turbofno_amd`.

A case is a spectral layer (or the steps of one, called one by one) of a given size. `kind` says how a user calls it:

  layer_1d   tf.layer_1d: the fused 1D layer, x[K][bs][DY] -> y[N][bs][DY]
  layer_2d   tf.layer_2d: the 2D layer, x[K][bs][DX][DY] -> y[N][bs][DX][DY], algorithm chosen by size
  steps_1d   the 1D layer as three calls, with the truncated spectra kept by the caller: fft_stride_DY, cgemm, ifft_stride_DY
  halves_1d  the 1D layer as forward transform with the product fused in (fused_fft_cgemm), then the product with a second
             weight matrix fused into the backward transform (fused_cgemm_ifft): two spectral mixings between one pair of
             transforms

All data are complex64 on the GPU. The caller keeps the output and workspace tensors between calls, as a training or serving
loop does. The sizes are those of benchmark_config/ (lengths 128 to 1024, 64 retained modes per axis, K = 8 ... 128 input
channels in steps of 8, N = 64 or 128 output channels, batches of 1 to 32768 signals or 1 to 128 images) and of bench.py.
"""
import math

import torch

import turbofno_amd as tf

MODES = tf.MODES
_LARGEST_BYTES = 8 * 32768 * 256 * (128 + 128) + 8 * 128 * 128      # the largest listed case


def listed():
    return [
        # a single signal through a narrow layer: latency of one call, nothing else
        dict(name="1d_single", kind="layer_1d", bs=1, DY=128, K=8, N=64, field=False),
        # a small training batch of a wide 1D operator (benchmark_config/large_hidden_1d.txt)
        dict(name="1d_wide_hidden", kind="layer_1d", bs=64, DY=256, K=128, N=128, field=True),
        # a training batch that is no power of two, channels that are no multiple of 16, the shorter length
        dict(name="1d_ragged", kind="layer_1d", bs=1000, DY=128, K=40, N=128, field=True),
        # 2^20 retained modes per channel: the size of the 1D channel sweep of the published charts
        dict(name="1d_million_modes", kind="layer_1d", bs=16384, DY=128, K=64, N=64, field=False),
        # the last line of the default 1D grid: the largest batch with the most channels, a throughput run
        dict(name="1d_largest", kind="layer_1d", bs=32768, DY=256, K=128, N=128, field=True),
        # long signals (time series of 1024 samples) in a batch that fills the GPU
        dict(name="1d_long_signal", kind="layer_1d", bs=2048, DY=1024, K=32, N=64, field=True),
        # the layer built from its separate steps, for callers that look at or change the spectra in between
        dict(name="1d_steps", kind="steps_1d", bs=1024, DY=256, K=64, N=64, field=True),
        # one field at a time: inference of a 2D operator
        dict(name="2d_single", kind="layer_2d", bs=1, DX=256, DY=256, K=16, N=64, field=True),
        # a small batch of fields that are not square
        dict(name="2d_small_batch", kind="layer_2d", bs=4, DX=128, DY=256, K=32, N=64, field=False),
        # a training batch of small fields with a widening layer, not a power of two
        dict(name="2d_ragged", kind="layer_2d", bs=40, DX=128, DY=128, K=72, N=128, field=False),
        # the workload of bench.py
        dict(name="2d_training", kind="layer_2d", bs=16, DX=256, DY=256, K=64, N=64, field=True),
        # a training batch of finely resolved fields
        dict(name="2d_fine_grid", kind="layer_2d", bs=16, DX=512, DY=512, K=32, N=64, field=True),
    ]


def _log_uniform(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5)))))))


def draw(rng):
    """One more case of the same ranges. Batch sizes are spread over their logarithm (any integer, odd ones among them)."""
    while True:
        kind = rng.choice(["layer_1d", "layer_1d", "layer_2d", "layer_2d", "layer_2d", rng.choice(["steps_1d", "halves_1d"])])
        case = dict(kind=kind, K=8 * rng.randint(1, 16), N=rng.choice([64, 64, 128]), field=rng.random() < 0.5)
        if kind == "layer_2d":
            case.update(bs=_log_uniform(rng, 1, 128), DX=rng.choice([128, 256, 256, 512, 1024]),
                        DY=rng.choice([128, 256, 256, 512, 1024]))
        else:
            case.update(bs=_log_uniform(rng, 1, 32768), DY=rng.choice([128, 256, 256, 512, 1024]))
        if work(case)["bytes"] <= _LARGEST_BYTES:
            return case


def _grid(case):
    return (case["DX"], case["DY"]) if case["kind"] == "layer_2d" else (case["DY"],)


def _inputs(case, gen, channels):
    """x[channels][bs][grid]. field: a Gaussian random field with power spectrum (|k|^2 + 9)^-2.5 and unit variance (the
    vorticity-like input of bench.py) plus 1 % of white noise; else real and imaginary parts uniform in [-1, 1]."""
    grid = _grid(case)
    x = torch.empty((channels, case["bs"]) + grid, dtype=torch.complex64, device="cuda")
    if case["field"]:
        k2 = sum(torch.meshgrid(*[torch.fft.fftfreq(d, 1.0 / d, device="cuda") ** 2 for d in grid], indexing="ij"))
        amp = (k2 + 9.0) ** -1.25
        amp = amp * (math.prod(grid) / torch.linalg.vector_norm(amp))      # unit variance after the 1/D of ifftn
    per_sample = math.prod(grid)
    chunk = max(1, (1 << 26) // per_sample)                                 # at most 2^26 values at a time
    for c in range(channels):
        for b in range(0, case["bs"], chunk):
            part = x[c, b:b + chunk]
            if case["field"]:
                white = torch.randn(part.shape, dtype=torch.complex64, device="cuda", generator=gen)
                part.copy_(torch.fft.ifftn(white * amp, dim=tuple(range(1, 1 + len(grid)))))
                part.add_(white, alpha=0.01)
            else:
                torch.view_as_real(part).uniform_(-1.0, 1.0, generator=gen)
    return x


def _weights(case, gen, rows, cols):
    """W[rows][cols]: complex normal, scaled so that the product keeps the variance of its input."""
    return torch.randn((rows, cols), dtype=torch.complex64, device="cuda", generator=gen) / math.sqrt(cols)


def _empty(*shape):
    return torch.empty(shape, dtype=torch.complex64, device="cuda")


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    kind, bs, K, N = case["kind"], case["bs"], case["K"], case["N"]
    st = dict(case=case, x=_inputs(case, gen, K), W=_weights(case, gen, N, K), y=_empty(N, bs, *_grid(case)))
    if kind == "layer_2d":
        need = tf.layer_2d_workspace_bytes(bs, case["DX"], case["DY"], K, N)
        st["workspace"] = torch.empty(need, dtype=torch.uint8, device="cuda")
    elif kind == "steps_1d":
        st["spectra"] = _empty(K, bs, MODES)
        st["product"] = _empty(N, bs, MODES)
    elif kind == "halves_1d":
        st["W2"] = _weights(case, gen, N, N)
        st["product"] = _empty(N, bs, MODES)
    return st


def run(state):
    case, x, W, y = state["case"], state["x"], state["W"], state["y"]
    kind = case["kind"]
    if kind == "layer_1d":
        return tf.layer_1d(x, W, y=y)
    if kind == "layer_2d":
        return tf.layer_2d(x, W, y=y, workspace=state["workspace"])
    K, N, M = case["K"], case["N"], MODES * case["bs"]
    product = state["product"]
    if kind == "steps_1d":
        spectra = state["spectra"]
        tf.fft_stride_DY(x, spectra, 8, K * case["bs"])
        tf.cgemm(M, N, K, spectra, W, product)
        tf.ifft_stride_DY(product, y, 8, N * case["bs"])
        return spectra, product, y
    tf.fused_fft_cgemm(M, N, K, x, W, product)
    tf.fused_cgemm_ifft(M, N, N, product, state["W2"], y)
    return product, y


def _fft_flops(length):
    """Real operations of one transform of `length` of which 64 values are kept (or given): full-length radix-2 stages on
    blocks of 64 and one multiply-add per sample for the folding onto them, the fewest known up to a small factor."""
    return length * (5.0 * math.log2(MODES) + 8.0)


def work(case):
    kind, bs, K, N = case["kind"], case["bs"], case["K"], case["N"]
    grid = _grid(case)
    points = math.prod(grid)
    modes = MODES ** len(grid)
    if kind == "layer_2d":
        per_field = case["DX"] * _fft_flops(case["DY"]) + MODES * _fft_flops(case["DX"])
    else:
        per_field = _fft_flops(case["DY"])
    nbytes = 8 * bs * points * (K + N) + 8 * K * N
    flops = per_field * bs * (K + N) + 8.0 * bs * modes * K * N
    if kind == "steps_1d":
        nbytes += 2 * 8 * bs * modes * (K + N)          # spectra and product: written by one step, read by the next
    elif kind == "halves_1d":
        nbytes += 2 * 8 * bs * modes * N + 8 * N * N    # the product between the two halves, the second weights
        flops += 8.0 * bs * modes * N * N
    return dict(bytes=int(nbytes), flops=flops)


def tolerance(case):
    """32-bit arithmetic throughout. Against a 64-bit evaluation: relative error 1.5e-7 to 4.1e-7 (largest for two products
    in a row), largest single error 5e-6 of the larger of value and root mean square (spectra of smooth fields)."""
    return {"rel": 1.6e-6, "max": 2e-5}
