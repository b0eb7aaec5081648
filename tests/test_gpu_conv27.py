"""The staged 3x3x3 convolution against the float64 oracle where its tiling
can go wrong: voxel counts at the edges of its tiles, dilations up to its
limit and beyond the grid, every channel combination, several tiles per
workgroup (GPU)."""
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
