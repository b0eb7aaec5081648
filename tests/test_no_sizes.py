"""Field-operator entries at channel counts without a kernel: zero and negative
ones are refused with an error code or do nothing, as they did before the
kernels were made for given channel counts."""
from __future__ import annotations

import ctypes as C

import pytest

from cudadsmc_amd import _capi

P, L, I = C.c_void_p, C.c_long, C.c_int
HERE = P(4096)  # never dereferenced: the calls below end on the host


def entry(name, *types):
    f = getattr(_capi.lib(), name)
    f.argtypes, f.restype = types, I
    return f


@pytest.mark.parametrize("cout", [0, -32])
def test_bias_gradients_refuse_no_channels(cout):
    plain = entry("dsmc_no_bias_grad", P, L, I, P, P, L, I, P)
    fused = entry("dsmc_no_relu_bias_bwd", P, P, P, L, I, P, P, L, I, P)
    assert plain(HERE, 10, cout, HERE, HERE, 100, 0, None) == -1
    assert fused(HERE, HERE, HERE, 10, cout, HERE, HERE, 100, 0, None) == -1
    assert plain(HERE, 0, cout, HERE, HERE, 100, 0, None) == 0  # no voxels: nothing to do


@pytest.mark.parametrize("taps", [1, 27])
@pytest.mark.parametrize("cin,cout", [(0, 32), (32, 0), (-32, 32), (32, -32)])
def test_weight_gradient_refuses_no_channels(cin, cout, taps):
    f = entry("dsmc_no_conv_bwd_w", P, P, P, P, L, *[I] * 10, P)
    assert f(HERE, HERE, HERE, HERE, 0, 1, 2, 2, 2, cin, cout, taps, 1, 64, 0, None) == -1


@pytest.mark.gpu
@pytest.mark.parametrize("taps", [1, 27])
def test_convolution_to_no_channels_writes_nothing(taps):
    torch = pytest.importorskip("torch")
    from cudadsmc_amd import neural

    x = torch.ones(8 * 32, dtype=torch.bfloat16, device="cuda")
    y = torch.full((4096,), 3.0, dtype=torch.bfloat16, device="cuda")
    neural.conv_fwd(x, x, None, 1, (2, 2, 2), 32, 0, taps, 1, y=y)
    assert bool((y == 3.0).all())
