"""The staged 3x3x3 convolution against the float64 oracle where its tiling
can go wrong: voxel counts at the edges of its tiles, dilations up to its
limit and beyond the grid, combinations of channels, several tiles per
workgroup (GPU). test_gpu_conv_forms.py has the forms of two weight buffers
and of two workgroups per CU."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import no_ref

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def bf(a: np.ndarray):
    return torch.from_numpy(no_ref.bf16_round(np.asarray(a, np.float32))).cuda().to(torch.bfloat16)


@pytest.mark.parametrize("B,shape,cin,cout,dil", [
    (1, (1, 1, 1), 32, 32, 1), (1, (2, 2, 31), 64, 96, 8), (1, (1, 8, 16), 96, 64, 1), (1, (1, 3, 43), 128, 128, 2),
    (2, (4, 8, 4), 32, 128, 4), (1, (5, 7, 37), 96, 96, 0), (3, (3, 5, 9), 128, 32, 8), (1, (9, 3, 19), 64, 64, 9),
    # one voxel above 128 tiles of 256: the wider tile, then more tiles than workgroups of it
    (1, (1, 331, 99), 96, 96, 3), (2, (11, 61, 103), 64, 32, 8)])
def test_staged_convolution(B, shape, cin, cout, dil):
    from cudadsmc_amd import neural

    print(f"conv27 B={B} shape={shape} cin={cin} cout={cout} dil={dil}", flush=True)
    rng = np.random.default_rng(cin + cout + dil)
    M = B * int(np.prod(shape))
    x = no_ref.bf16_round(rng.standard_normal((B,) + shape + (cin,)).astype(np.float32))
    w = no_ref.bf16_round((rng.standard_normal((27, cout, cin)) / np.sqrt(27 * cin)).astype(np.float32))
    b = rng.standard_normal(cout).astype(np.float32)
    res = no_ref.bf16_round(rng.standard_normal((M, cout)).astype(np.float32))
    guard = 64  # elements past the end must stay as they are
    y = torch.full((M * cout + guard,), 3.0, dtype=torch.bfloat16, device="cuda")
    h, y32 = torch.full_like(y, 3.0), torch.full((M * cout + guard,), 3.0, device="cuda")
    neural.conv_fwd(bf(x).reshape(M, cin), bf(w), torch.from_numpy(b).cuda(), B, shape, cin, cout, 27, dil, relu=True,
                    res=bf(res), y=y, y32=y32, h=h)
    hw = np.maximum(no_ref.conv(x, w, b, dil).reshape(M, cout), 0.0)
    yw = hw + res.astype(np.float64)
    got = {k: t.float().cpu().numpy() for k, t in (("y", y), ("h", h), ("y32", y32))}
    for a in got.values():
        assert np.all(a[M * cout:] == 3.0)
    gy, gh, g32 = (got[k][:M * cout].reshape(M, cout) for k in ("y", "h", "y32"))
    # FP32 accumulation of 27 cin products of order 1 / sqrt(27 cin): far below 2e-5 of the largest value;
    # the BF16 outputs add one rounding (2^-8 relative) to that
    acc = 2e-5 * max(np.max(np.abs(hw)), 1e-30)
    assert np.max(np.abs(g32 - yw)) <= acc + 2.0 ** -23 * np.max(np.abs(yw))
    assert np.all(np.abs(gh - hw) <= 2.0 ** -8 * np.abs(hw) + acc)
    assert np.all(np.abs(gy - yw) <= 2.0 ** -8 * np.abs(yw) + 2 * acc)


@pytest.mark.parametrize("B,shape,cin,cout,dil,chunk", [
    (1, (1, 1, 1), 32, 32, 1, 64), (1, (2, 3, 37), 64, 128, 8, 64), (2, (5, 7, 11), 128, 96, 2, 128),
    (1, (4, 1, 17), 128, 128, 0, 64), (3, (3, 5, 9), 96, 32, 4, 4096), (1, (9, 3, 19), 32, 64, 9, 64),
    # many voxels in a partial, and enough of them for two workgroups per CU
    (1, (40, 50, 51), 32, 96, 3, 65536), (1, (40, 50, 51), 64, 32, 8, 1024), (2, (60, 50, 51), 32, 32, 1, 2048)])
def test_staged_weight_gradient(B, shape, cin, cout, dil, chunk):
    from cudadsmc_amd import neural

    print(f"conv27 weight gradient B={B} shape={shape} cin={cin} cout={cout} dil={dil} chunk={chunk}", flush=True)
    rng = np.random.default_rng(cin + cout + dil)
    M = B * int(np.prod(shape))
    x = no_ref.bf16_round(rng.standard_normal((B,) + shape + (cin,)).astype(np.float32))
    dy = no_ref.bf16_round(rng.standard_normal((B,) + shape + (cout,)).astype(np.float32))
    n = 27 * cout * cin
    part = torch.full(((M + chunk - 1) // chunk * n,), float("nan"), device="cuda")  # no partial may be read unwritten
    dw = torch.full((27, cout, cin), 7.0, device="cuda")
    want = no_ref.conv_grad_w(x, dy, 27, dil)
    for times, accumulate in ((1, False), (2, True)):
        neural.conv_bwd_w(bf(x).reshape(M, cin), bf(dy).reshape(M, cout), dw, part, B, shape, cin, cout, 27, dil,
                          chunk=chunk, accumulate=accumulate)
        got = dw.cpu().numpy()
        # FP32 accumulation, as in the tests of the general kernel: 2e-5 of the largest value
        assert np.max(np.abs(got - times * want)) <= 2e-5 * np.max(np.abs(times * want))


@pytest.mark.parametrize("M,cout,skew", [(1, 32, 0), (513, 128, 0), (1000, 96, 1), (4097, 64, 0), (70001, 96, 0)])
def test_relu_and_bias_gradient_in_one_pass(M, cout, skew):
    """Against the two separate kernels (the same values and sums) and the
    float64 sums; skew: arrays that are not 16-byte aligned."""
    from cudadsmc_amd import neural

    rng = np.random.default_rng(M)
    dy, h = (bf(rng.standard_normal(M * cout + skew))[skew:] for _ in range(2))
    dz, dz2 = (torch.full((M * cout + skew,), 5.0, dtype=torch.bfloat16, device="cuda")[skew:] for _ in range(2))
    part = torch.full(((M + 511) // 512 * cout,), float("nan"), device="cuda")
    db, db2 = torch.zeros(cout, device="cuda"), torch.zeros(cout, device="cuda")
    neural.relu_bias_bwd(dy, h, dz, M, cout, db, part)
    neural.relu_bwd(dy, h, dz2)
    neural.bias_grad(dz2, M, cout, db2, part)
    want = torch.where(h > 0, dy, torch.zeros_like(dy))
    assert torch.equal(dz, want) and torch.equal(dz2, want) and torch.equal(db, db2)
    exact = want.double().reshape(M, cout).sum(0)
    # FP32 sums of M BF16 values in chains of at most 64 and their partials
    assert float((db.double() - exact).abs().max()) <= 1e-6 * float(want.double().abs().reshape(M, cout).sum(0).max())


@pytest.mark.parametrize("M,cin,cout", [(1, 32, 32), (33, 96, 32), (127, 32, 96), (5000, 64, 128), (140001, 128, 64)])
def test_pointwise_convolution(M, cin, cout):
    from cudadsmc_amd import neural

    rng = np.random.default_rng(M + cin)
    x, w = bf(rng.standard_normal((M, cin))), bf(rng.standard_normal((1, cout, cin)) / np.sqrt(cin))
    y32 = torch.full((M * cout + 64,), 3.0, device="cuda")
    neural.conv_fwd(x, w, None, 1, (1, 1, M), cin, cout, 1, 1, y32=y32)
    want = x.double() @ w[0].double().T
    # FP32 accumulation of at most 128 products
    assert float((y32[:M * cout].reshape(M, cout).double() - want).abs().max()) <= 2e-5 * float(want.abs().max())
    assert bool((y32[M * cout:] == 3.0).all())


# workgroups per 32 input channels up to 1024 of them, then one for all channels
@pytest.mark.parametrize("M,cin,cout,chunk", [(1, 128, 32, 64), (1000, 96, 128, 128), (64 * 256, 128, 32, 64),
                                              (64 * 256 + 1, 128, 32, 64)])
def test_one_tap_weight_gradient(M, cin, cout, chunk):
    from cudadsmc_amd import neural

    print(f"one-tap weight gradient M={M} cin={cin} cout={cout} chunk={chunk}", flush=True)
    rng = np.random.default_rng(M + cin)
    x = no_ref.bf16_round(rng.standard_normal((M, cin)).astype(np.float32))
    dy = no_ref.bf16_round(rng.standard_normal((M, cout)).astype(np.float32))
    part = torch.full(((M + chunk - 1) // chunk * cin * cout,), float("nan"), device="cuda")
    dw = torch.full((1, cout, cin), 7.0, device="cuda")
    want = dy.astype(np.float64).T @ x.astype(np.float64)
    neural.conv_bwd_w(bf(x), bf(dy), dw, part, 1, (1, 1, M), cin, cout, 1, 1, chunk=chunk, accumulate=False)
    # FP32 accumulation, as above
    assert np.max(np.abs(dw.cpu().numpy()[0] - want)) <= 2e-5 * np.max(np.abs(want))
