"""The scorer's forward kernel against the forward pass inside its gradient kernel, bit for bit: the
gradient reads gathered tiles, the forward the same tiles in place, at every alignment that an
origin and a row stride can give, with more tiles than work groups and out-of-range origins
among them; and the gradient's reduction over part counts around its blocks of rows."""

import ctypes

import numpy as np
import pytest

from oracle import scorer as sc

pytestmark = pytest.mark.gpu


def params(seed):
    rng = np.random.default_rng(seed)
    return sc.init_params(rng) + 0.1 * rng.standard_normal(sc.init_params(rng).shape)


@pytest.mark.parametrize('dtype', ['float32', 'float16', 'bfloat16'])
@pytest.mark.parametrize('stride', [700, 701])
@pytest.mark.parametrize('n', [1, 3, 1100])
def test_forward_in_place_equals_gradient_forward(dtype, stride, n):
    import torch
    import pirate_amd as pa
    from pirate_amd import _lib as L
    print(f'[scorer tiles] {dtype} stride {stride} n {n}', flush=True)
    rng = np.random.default_rng(n)
    B, R, T = 2, 200, 690
    buf = torch.from_numpy(rng.standard_normal(B * R * stride + 3).astype(np.float32)).cuda().to(getattr(torch, dtype))
    rows = buf[3:].view(B, R, stride)                          # rows start off any alignment
    src = pa.TileSource(L.TileSource(ctypes.c_void_p(rows.data_ptr()), ['float32', 'float16', 'bfloat16'].index(dtype),
                                     B, R * stride, R, stride, 2, T, None), [buf])
    o = np.stack([rng.integers(0, B, n), rng.integers(0, R - 63, n), rng.integers(2, T - 255, n)], axis=1).astype(np.int32)
    o[:, 2][::4] &= ~3                                        # some aligned
    tiles = torch.stack([rows[b, r:r + 64, t:t + 256] for b, r, t in o]).contiguous()
    bad = np.arange(n) % 7 == 5
    o[bad, 1] = R - 63                                         # one row too far
    bad |= o[:, 2] < 2                                         # before t_lo
    scr = pa.LearnedScorer(params(5))
    got = scr.forward(src.with_origins(o)).cpu().numpy()
    want = scr.grad(tiles, torch.zeros(n))[1].cpu().numpy()
    assert np.all(np.isnan(got[bad]))
    np.testing.assert_array_equal(got[~bad], want[~bad])


@pytest.mark.parametrize('n', [1, 255, 256, 257])
def test_gradient_reduction(n):
    import torch
    import pirate_amd as pa
    rng = np.random.default_rng(n)
    theta = params(7)
    x = rng.standard_normal((n, sc.C0, sc.T)).astype(np.float32)
    y = (rng.random(n) < 0.5).astype(np.float32)
    scr = pa.LearnedScorer(theta)
    g = sc.unpack(scr.grad(torch.from_numpy(x).cuda(), torch.from_numpy(y))[0].cpu().numpy().astype(np.float64))
    want = sc.unpack(sc.loss_and_grad(theta, x.astype(np.float64), y, rounding='bf16')[1])
    for name, _ in sc.SHAPES:        # the tolerance of float32 sums and rare bf16 rounding flips
        scale = max(np.max(np.abs(want[name])), 1e-30)
        assert np.max(np.abs(g[name] - want[name])) <= 2e-3 * scale, name
