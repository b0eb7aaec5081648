"""The staged convolutions in the forms that large layers of wide channels
take, on arrays at any alignment, on infinities and NaN, and in place (GPU).

A call whose arrays are not 16-byte aligned goes to the general kernels, which
add in the same order: the staged ones must give the same bits."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import no_ref
from test_gpu_conv27 import bf

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

SKEW = 2  # elements: 4 bytes for BF16 and 8 for FP32, so that vector loads of the general kernels stay legal


def skewed(t):
    """The same values, not 16-byte aligned."""
    out = torch.empty(t.numel() + SKEW, dtype=t.dtype, device=t.device)[SKEW:]
    out.copy_(t.reshape(-1))
    assert out.data_ptr() % 16 != 0
    return out


def same(a, b) -> bool:
    """Bit for bit, but any NaN for any NaN."""
    nan = torch.isnan(a)
    return torch.equal(nan, torch.isnan(b)) and torch.equal(a[~nan], b[~nan])


def layer(M, cin, cout, taps, seed):
    rng = np.random.default_rng(seed)
    x = no_ref.bf16_round(rng.standard_normal((M, cin)).astype(np.float32))
    w = no_ref.bf16_round((rng.standard_normal((taps, cout, cin)) / np.sqrt(taps * cin)).astype(np.float32))
    res = no_ref.bf16_round(rng.standard_normal((M, cout)).astype(np.float32))
    return x, w, rng.standard_normal(cout).astype(np.float32), res


def forward(x, w, b, res, shape, cin, cout, taps, dil, y=None, relu=True):
    from cudadsmc_amd import neural

    M = int(np.prod(shape))
    y = torch.full((M * cout,), 3.0, dtype=torch.bfloat16, device="cuda") if y is None else y
    h, y32 = torch.full((M * cout,), 3.0, dtype=torch.bfloat16, device="cuda"), torch.full((M * cout,), 3.0, device="cuda")
    neural.conv_fwd(x, w, b, 1, shape, cin, cout, taps, dil, relu=relu, res=res, y=y, y32=y32, h=h)
    return y, h, y32


# 32769 voxels: two voxel tiles per wave; with 128 input channels and 96 or 128 output channels only two weight buffers
# fit. 140400 voxels: 549 tiles of 256, so that some of the (at most 256) workgroups take three
@pytest.mark.parametrize("shape,cin,cout,dil", [((1, 331, 99), 128, 128, 1), ((33, 1, 993), 128, 96, 8),
                                                ((60, 45, 52), 128, 128, 2)])
def test_two_weight_buffers(shape, cin, cout, dil):
    print(f"two weight buffers shape={shape} cin={cin} cout={cout} dil={dil}", flush=True)
    M = int(np.prod(shape))
    x, w, b, res = layer(M, cin, cout, 27, 7)
    dev = bf(x), bf(w), torch.from_numpy(b).cuda(), bf(res)
    y, h, y32 = forward(*dev, shape, cin, cout, 27, dil)
    for got, want in zip((y, h, y32), forward(skewed(dev[0]), *dev[1:], shape, cin, cout, 27, dil)):
        assert torch.equal(got, want)
    hw = np.maximum(no_ref.conv(x.reshape((1,) + shape + (cin,)), w, b, dil).reshape(M, cout), 0.0)
    yw = hw + res.astype(np.float64)
    # FP32 accumulation of 27 cin products of order 1 / sqrt(27 cin): far below 2e-5 of the largest value
    got = y32.cpu().numpy().reshape(M, cout)
    assert np.max(np.abs(got - yw)) <= 2e-5 * np.max(np.abs(hw)) + 2.0 ** -23 * np.max(np.abs(yw))


# more than 256 items of a chunk of voxels and four taps: two workgroups per CU share its LDS. 41 chunks of several
# blocks of 32 voxels, the last one ragged
@pytest.mark.parametrize("cin,cout,chunk", [(96, 96, 256), (64, 64, 128), (64, 96, 256), (32, 128, 192)])
def test_two_workgroups_per_cu_weight_gradient(cin, cout, chunk):
    from cudadsmc_amd import neural

    print(f"paired weight gradient cin={cin} cout={cout} chunk={chunk}", flush=True)
    shape = (1, 41, chunk - 3)
    M = int(np.prod(shape))
    chunks = (M + chunk - 1) // chunk
    assert chunks * 7 > 256 and M % 32
    x, _, _, dy = layer(M, cin, cout, 27, cin + cout)
    part = torch.full((chunks * 27 * cout * cin,), float("nan"), device="cuda")
    dw = torch.full((27, cout, cin), 7.0, device="cuda")
    neural.conv_bwd_w(bf(x), bf(dy), dw, part, 1, shape, cin, cout, 27, 3, chunk=chunk)
    want = no_ref.conv_grad_w(x.reshape((1,) + shape + (cin,)), dy.reshape((1,) + shape + (cout,)), 27, 3)
    # FP32 accumulation, as in the tests of the general kernel: 2e-5 of the largest value
    assert np.max(np.abs(dw.cpu().numpy() - want)) <= 2e-5 * np.max(np.abs(want))


@pytest.mark.parametrize("taps,shape,cin,cout", [(27, (3, 9, 37), 96, 64), (1, (1, 1, 999), 64, 96)])
def test_unaligned_forward(taps, shape, cin, cout):
    """Each array in turn 4 or 8 bytes off."""
    M = int(np.prod(shape))
    x, w, b, res = layer(M, cin, cout, taps, 3)
    x, w, b, res = bf(x), bf(w), torch.from_numpy(b).cuda(), bf(res)
    want = forward(x, w, b, res, shape, cin, cout, taps, 2)
    for args in ((skewed(x), w, b, res), (x, skewed(w), b, res), (x, w, skewed(b), res), (x, w, b, skewed(res))):
        for got, ref in zip(forward(*args, shape, cin, cout, taps, 2), want):
            assert torch.equal(got, ref)
    y = torch.empty(M * cout + SKEW, dtype=torch.bfloat16, device="cuda")[SKEW:]
    for got, ref in zip(forward(x, w, b, res, shape, cin, cout, taps, 2, y=y), want):
        assert torch.equal(got, ref)


@pytest.mark.parametrize("taps", [1, 27])
def test_output_in_place_of_the_residual(taps):
    shape, cin, cout = (4, 9, 37), 64, 96
    x, w, b, res = layer(int(np.prod(shape)), cin, cout, taps, 5)
    x, w, b, res = bf(x), bf(w), torch.from_numpy(b).cuda(), bf(res).reshape(-1)
    want = forward(x, w, b, res, shape, cin, cout, taps, 1)
    got = forward(x, w, b, res, shape, cin, cout, taps, 1, y=res)
    assert got[0].data_ptr() == res.data_ptr()
    for a, ref in zip(got, want):
        assert torch.equal(a, ref)


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("row", [0, -1])
def test_infinities_and_nan_stay_where_they_are(bad, row):
    """The first rows are what the staged kernels load in place of rows outside
    the arrays, and the last ones lie beside the rows past the end."""
    from cudadsmc_amd import neural

    shape, cin, cout, chunk = (3, 7, 33), 64, 96, 64
    M = int(np.prod(shape))
    assert M % 64
    x, w, b, dy = layer(M, cin, cout, 27, 9)
    x, w, b, dy = bf(x), bf(w), torch.from_numpy(b).cuda(), bf(dy)
    chunks = (M + chunk - 1) // chunk
    for x_bad, dy_bad in ((True, False), (False, True)):
        xx, dd = x.clone(), dy.clone()
        if x_bad:
            xx[row, 5] = bad
        if dy_bad:
            dd[row, 11] = bad
        out = []
        for sx, sdy in ((xx, dd), (skewed(xx), skewed(dd))):
            part = torch.full((chunks * 27 * cout * cin,), 0.0, device="cuda")
            dw = torch.zeros((27, cout, cin), device="cuda")
            neural.conv_bwd_w(sx, sdy, dw, part, 1, shape, cin, cout, 27, 2, chunk=chunk)
            out.append((dw,) + forward(sx, w, b, sdy, shape, cin, cout, 27, 2, relu=False))  # a ReLU would drop the NaN
        for got, want in zip(*out):
            assert same(got, want)
        dw, _, h, _ = out[0]
        off = (~torch.isfinite(dw)).any(0)  # [cout][cin]
        spread = off.any(0).nonzero().flatten() if x_bad else off.any(1).nonzero().flatten()
        assert spread.tolist() == [5 if x_bad else 11]
        if x_bad:  # 27 voxels of the grid see it at most, and not all of them lie in the grid
            assert 0 < int((~torch.isfinite(h.reshape(M, cout))).any(1).sum()) <= 27


# a wave has two chunks of 512 voxels at 32 channels, one else; ragged in the first and the second of them
@pytest.mark.parametrize("M", [1, 511, 513, 1000, 1537, 4600])
@pytest.mark.parametrize("cout", [32, 96])
def test_bias_gradient_of_a_ragged_chunk(M, cout):
    """The sums of a ragged last chunk are those of the chunk filled up with
    zeros, bit for bit, and nothing is written past the end."""
    from cudadsmc_amd import neural

    rng = np.random.default_rng(M + cout)
    chunks = (M + 511) // 512
    dy, h = (bf(rng.standard_normal((chunks * 512, cout))) for _ in range(2))
    dy[M:] = 0.0
    dz = torch.full((chunks * 512, cout), 5.0, dtype=torch.bfloat16, device="cuda")
    part = torch.full((chunks * cout,), float("nan"), device="cuda")
    out = [torch.zeros(cout, device="cuda") for _ in range(4)]
    neural.bias_grad(dy, M, cout, out[0], part)
    neural.bias_grad(dy, chunks * 512, cout, out[1], part)
    neural.relu_bias_bwd(dy, h, dz, M, cout, out[2], part)
    assert bool((dz[M:] == 5.0).all())
    assert torch.equal(dz[:M], torch.where(h[:M] > 0, dy[:M], torch.zeros_like(dy[:M])))
    dz[M:] = 0.0
    neural.bias_grad(dz, chunks * 512, cout, out[3], part)
    assert torch.equal(out[0], out[1]) and torch.equal(out[2], out[3])
