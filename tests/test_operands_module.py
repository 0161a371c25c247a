"""The compiled operand checks of the binding (csrc/operands.cpp) against the checks in Python: what one takes the other takes, with the same
values, what one refuses the other refuses with the same error."""
import sysconfig
import types

import numpy as np
import pytest
import torch

import turbofno_amd as tf
from turbofno_amd import api

needs_module = pytest.mark.skipif(api._operands is None, reason="extension not built")


def _c64(*shape, device):
    return torch.zeros(shape, dtype=torch.complex64, device=device)


def _forms(device):
    """(name, call): every call site of the module, with operands right and wrong in one respect each"""
    z = lambda *s: _c64(*s, device=device)
    K, S, D, N = 8, 2, 128, 64
    x, W, y = z(K, S, D), z(N, K), z(N, S, D)
    x2, y2 = z(K, 1, 128, 128), z(N, 1, 128, 128)
    ws = torch.zeros(tf.layer_2d_workspace_bytes(1, 128, 128, K, N), dtype=torch.uint8, device=device)
    wide = z(K, S, 2 * D)
    one = [
        ("plain", (x, W, y), {}), ("parameter", (torch.nn.Parameter(x), W, y), {}), ("view", (wide.view(-1)[:K * S * D].view(K, S, D), W, y), {}),
        ("offset by one value", (wide.view(-1)[1:1 + K * S * D].view(K, S, D), W, y), {}), ("strided", (wide[:, :, ::2], W, y), {}),
        ("transposed W", (x, z(K, N).t(), y), {}), ("double", (x.to(torch.complex128), W, y), {}), ("real", (x.real.contiguous(), W, y), {}),
        ("two dimensions", (x.view(K, S * D), W, y), {}), ("W of other K", (x, z(N, K + 8), y), {}), ("y of other N", (x, W, z(2 * N, S, D)), {}),
        ("K no multiple of 8", (z(4, S, D), z(N, 4), y), {}), ("length not built", (z(K, S, 200), W, z(N, S, 200)), {}), ("array", (np.zeros((K, S, D), np.complex64), W, y), {}),
        ("alpha real", (x, W, y), dict(alpha=2)), ("alpha text", (x, W, y), dict(alpha="1+2j")), ("alpha wrong", (x, W, y), dict(alpha="one")), ("alpha none", (x, W, y), dict(alpha=None)),
        ("dimX", (x, W, y), dict(dimX=2)), ("dimX no divisor", (x, W, y), dict(dimX=3)), ("dimX zero", (x, W, y), dict(dimX=0)), ("dimX numpy", (x, W, y), dict(dimX=np.int64(2))),
        ("no y", (x, W), {}), ("no signals", (z(K, 0, D), W, z(N, 0, D)), {}), ("conjugate view", (x.conj(), W, y), {}),
    ]
    two = [
        ("plain", (x2, W, y2), dict(workspace=ws)), ("small workspace", (x2, W, y2), dict(workspace=ws[:-256])), ("no workspace", (x2, W, y2), {}),
        ("float workspace", (x2, W, y2), dict(workspace=ws.float())), ("misaligned workspace", (x2, W, y2), dict(workspace=ws[8:])),
        ("strided workspace", (x2, W, y2), dict(workspace=ws[::2])), ("algo 9", (x2, W, y2), dict(workspace=ws, algo=9)), ("algo -1", (x2, W, y2), dict(workspace=ws, algo=-1)),
        ("y transposed", (x2, W, y2.transpose(2, 3)), dict(workspace=ws)), ("W of other K", (x2, z(N, 16), y2), dict(workspace=ws)),
    ]
    M = 64 * S
    A, C = z(K, M), z(N, M)
    rest = [
        ("cgemm", lambda: tf.cgemm(M, N, K, A, W, C)), ("cgemm sizes", lambda: tf.cgemm(M, N, K + 8, A, W, C)), ("cgemm strided", lambda: tf.cgemm(M // 2, N, K, A[:, ::2], W, C)),
        ("cgemm float size", lambda: tf.cgemm(float(M), N, K, A, W, C)),
        ("fused", lambda: tf.fused_fft_cgemm_ifft(M, N, K, x, W, y)), ("fused sizes", lambda: tf.fused_fft_cgemm_ifft(2 * M, N, K, x, W, y)),
        ("first half", lambda: tf.fused_fft_cgemm(M, N, K, x, W, C)), ("second half", lambda: tf.fused_cgemm_ifft(M, N, K, A, W, y)),
        ("second half sizes", lambda: tf.fused_cgemm_ifft(M, N, K, A, W, y[:, :1])), ("forward", lambda: tf.fft_stride_DY(x, z(K * S, 64), 8, K * S)),
        ("forward sizes", lambda: tf.fft_stride_DY(x, z(K * S, 32), 8, K * S)), ("backward", lambda: tf.ifft_stride_DY(z(K * S, 64), x, 8, K * S)),
        ("X axis", lambda: tf.fft_stride(x2, z(K, 64, 128), 8, 128, 128 * K)), ("X axis back", lambda: tf.ifft_stride(z(K, 64, 128), x2, 8, 128, 128 * K)),
        ("X axis sizes", lambda: tf.fft_stride(x2, z(K, 64, 64), 8, 128, 128 * K)),
    ]
    forms = [("1d " + n, (lambda a=a, k=k: tf.layer_1d(*a, **k))) for n, a, k in one] + [("2d " + n, (lambda a=a, k=k: tf.layer_2d(*a, **k))) for n, a, k in two]
    return forms + rest


def _outcome(call):
    try:
        return "returned", tuple(call().shape)
    except Exception as e:
        return type(e), str(e)


def _compare(device, monkeypatch):
    for name, call in _forms(device):
        print("form", name, flush=True)
        with_module = _outcome(call)
        with monkeypatch.context() as m:
            m.setattr(api, "_operands", None)
            without = _outcome(call)
        assert with_module == without, name


def test_a_module_of_another_torch_is_left_alone():
    """it would read tensors at the offsets of another build's headers"""
    here = "torch %s, %s" % (torch.__version__, sysconfig.get_config_var("SOABI"))
    module = types.SimpleNamespace(built_for=here)
    assert api._of_this_torch(module) is module
    for other in ("torch 2.9.0, " + sysconfig.get_config_var("SOABI"), "torch %s, cpython-311-x86_64-linux-gnu" % torch.__version__, "", None):
        assert api._of_this_torch(types.SimpleNamespace(built_for=other)) is None, other
    assert api._of_this_torch(types.SimpleNamespace()) is None         # built before the module named its torch


@needs_module
def test_the_built_module_names_its_torch():
    assert api._operands.built_for == "torch %s, %s" % (torch.__version__, sysconfig.get_config_var("SOABI"))


@needs_module
def test_same_refusals_without_a_gpu(monkeypatch):
    _compare("cpu", monkeypatch)


@needs_module
@pytest.mark.gpu
def test_same_forms_taken_and_refused(monkeypatch):
    """zeros in: every call either runs (the kernels accept the form) or raises before a launch"""
    _compare("cuda", monkeypatch)
    torch.cuda.synchronize()


@needs_module
@pytest.mark.gpu
def test_module_takes_the_plain_call():
    """the short way is the one that runs: status 0, the operands' own addresses, None or -1 for what is left to Python"""
    x, W, y = _c64(8, 2, 128, device="cuda"), _c64(64, 8, device="cuda"), _c64(64, 2, 128, device="cuda")
    tf.lib()
    assert api._operands.layer_1d(api._LAYER_1D, x, W, y, 1 + 0j, 1, api._stream()) == 0
    assert api._operands.layer_1d(api._LAYER_1D, x.cpu(), W, y, 1 + 0j, 1, api._stream()) == -1
    assert api._operands.operands(x, x.numel(), y, y.numel()) == (x.data_ptr(), y.data_ptr())
    assert api._operands.operands(x, x.numel() + 1) is None
    torch.cuda.synchronize()


def _random(*shape):
    gen = torch.Generator(device="cuda").manual_seed(len(shape) + shape[0])
    return torch.view_as_complex(torch.rand(shape + (2,), device="cuda", generator=gen) * 2 - 1)


def _values(call, y):
    y.fill_(float("nan"))
    call()
    return torch.view_as_real(y).clone()


@needs_module
@pytest.mark.gpu
def test_same_values_either_way(monkeypatch):
    """the same launch with the same arguments: alpha's parts, dimX, the algorithm and the workspace, bit for bit"""
    alpha, K, N = 0.5 - 0.75j, 16, 64
    W = _random(N, K)
    x, y = _random(K, 6, 256), torch.empty((N, 6, 256), dtype=torch.complex64, device="cuda")
    calls = [("layer_1d dimX=%d" % d, lambda d=d: tf.layer_1d(x, W, y=y, alpha=alpha, dimX=d), y) for d in (1, 2)]
    x2, y2 = _random(K, 2, 128, 256), torch.empty((N, 2, 128, 256), dtype=torch.complex64, device="cuda")
    for algo in (0, 1, 2, 3):
        ws = torch.zeros(tf.layer_2d_workspace_bytes(2, 128, 256, K, N, algo), dtype=torch.uint8, device="cuda")
        calls.append(("layer_2d algo=%d" % algo, lambda algo=algo, ws=ws: tf.layer_2d(x2, W, y=y2, alpha=alpha, workspace=ws, algo=algo), y2))
    M = 64 * 6
    A, C = _random(K, M), torch.empty((N, M), dtype=torch.complex64, device="cuda")
    calls += [("cgemm", lambda: tf.cgemm(M, N, K, A, W, C, alpha), C), ("fused", lambda: tf.fused_fft_cgemm_ifft(M, N, K, x, W, y, alpha), y),
              ("first half", lambda: tf.fused_fft_cgemm(M, N, K, x, W, C, alpha), C), ("second half", lambda: tf.fused_cgemm_ifft(M, N, K, A, W, y, alpha), y)]
    results = {}
    for name, call, out in calls:
        print("values", name, flush=True)
        short = _values(call, out)
        with monkeypatch.context() as m:
            m.setattr(api, "_operands", None)
            long = _values(call, out)
        assert not bool(torch.isnan(short).any()), name
        assert torch.equal(short, long), name
        results[name] = short
    # the algorithms round differently: a call that ran another one would show
    layers = [results["layer_2d algo=%d" % a] for a in (1, 2, 3)]
    assert not torch.equal(layers[0], layers[1]) and not torch.equal(layers[1], layers[2]) and not torch.equal(layers[0], layers[2])
