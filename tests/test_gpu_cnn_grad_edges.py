"""Weight-gradient kernels of the prior at the edges of their tiles: small
integers, where every product and partial sum is exact in FP32, so each kernel
must equal the FP64 sum over pixels bit for bit."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# widths around a 4-pixel step, a 32-pixel tile and a 64-pixel chunk; single rows and columns
SHAPES = [(1, 1, 1), (1, 1, 3), (2, 3, 4), (1, 2, 31), (1, 5, 33), (3, 2, 63), (1, 7, 65), (2, 70, 36), (1, 3, 129)]


def _shift_sums(img, act):
    """[9][ci] sums over p of img[p + off_t] act[p], zero outside the image."""
    B, H, W = img.shape
    p = np.pad(img, ((0, 0), (1, 1), (1, 1)))
    return np.stack([np.einsum("bhw,bhwc->c", p[:, t // 3:t // 3 + H, t % 3:t % 3 + W], act) for t in range(9)])


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("mode", [0, 1])
def test_narrow_gradients(shape, mode):
    from reconnet_amd.cnn import _p, _sigs, _st

    B, H, W = shape
    rng = np.random.default_rng(100 * W + 10 * H + mode)
    img = rng.integers(-3, 4, shape).astype(np.float64)
    act = rng.integers(-3, 4, shape + (32,)).astype(np.float64)
    x = torch.from_numpy(img).float().cuda()
    a = torch.from_numpy(act).cuda().to(torch.bfloat16)
    g = torch.full((320,), 7.0, device="cuda")     # mode 1 writes 289 entries and no more
    assert _sigs().rn_cnn_wgrad_narrow(_p(x), _p(a), _p(g), B, H, W, mode, _st()) == 0
    g = g.cpu().double().numpy()
    want = _shift_sums(img, act)
    # mode 1: the tensor is shifted instead, the image's shifts in reverse
    assert np.array_equal(g[:288].reshape(9, 32), want if mode == 0 else want[::-1])
    if mode == 0:
        assert np.array_equal(g[288:], act.sum((0, 1, 2)))
    else:
        assert g[288] == img.sum() and (g[289:] == 7.0).all()


@pytest.mark.parametrize("shape", SHAPES + [(5, 300, 40)])    # the last: several 64-row items per strip
def test_mid_gradients(shape):
    from reconnet_amd.cnn import _p, _sigs, _st

    B, H, W = shape
    rng = np.random.default_rng(100 * W + 10 * H + 5)
    a = rng.integers(-2, 3, shape + (32,)).astype(np.float64)
    d = rng.integers(-2, 3, shape + (32,)).astype(np.float64)
    at, dt = (torch.from_numpy(v).cuda().to(torch.bfloat16) for v in (a, d))
    g, gb = torch.empty(9, 32, 32, device="cuda"), torch.empty(32, device="cuda")
    assert _sigs().rn_cnn_wgrad_mid_bias(_p(at), _p(dt), _p(g), _p(gb), B, H, W, _st()) == 0
    p = np.pad(a, ((0, 0), (1, 1), (1, 1), (0, 0)))
    want = np.stack([np.tensordot(d, p[:, t // 3:t // 3 + H, t % 3:t % 3 + W], ((0, 1, 2), (0, 1, 2)))
                     for t in range(9)])
    assert np.array_equal(g.cpu().double().numpy(), want)
    assert np.array_equal(gb.cpu().double().numpy(), d.sum((0, 1, 2)))


@pytest.mark.parametrize("shape", [(1, 3, 4), (2, 5, 70), (1, 66, 33)])
@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_narrow_gradients_of_taps_off_the_image(shape, mode, bad):
    # a NaN or an infinity of one channel on the image's border reaches the taps whose
    # image pixel exists and no others; those keep their exact sums
    from reconnet_amd.cnn import _p, _sigs, _st

    B, H, W = shape
    rng = np.random.default_rng(W + mode)
    img = rng.integers(1, 4, shape).astype(np.float64)
    act = rng.integers(-3, 4, shape + (32,)).astype(np.float64)
    for y, x, c in ((0, 0, 5), (H - 1, W - 1, 8), (H // 2, 0, 31), (0, W // 2, 0)):
        a0, ok = act.copy(), np.zeros(shape)
        a0[B - 1, y, x, c], ok[B - 1, y, x] = 0.0, 1.0
        want = _shift_sums(img, a0)
        inside = _shift_sums(np.ones(shape), ok[..., None])[:, 0] > 0      # taps whose image pixel exists
        a1 = act.copy()
        a1[B - 1, y, x, c] = bad
        g = torch.empty(320, device="cuda")
        xt, at = torch.from_numpy(img).float().cuda(), torch.from_numpy(a1).cuda().to(torch.bfloat16)
        assert _sigs().rn_cnn_wgrad_narrow(_p(xt), _p(at), _p(g), B, H, W, mode, _st()) == 0
        got = g.cpu().double().numpy()[:288].reshape(9, 32)
        if mode == 1:
            got = got[::-1]
        assert not np.isfinite(got[inside, c]).any(), (y, x)
        got[inside, c] = want[inside, c]
        assert np.array_equal(got, want), (y, x)


@pytest.mark.parametrize("shape,row", [((1, 3, 32), 2), ((2, 70, 36), 69), ((1, 70, 36), 8), ((1, 70, 36), 7)])
def test_mid_gradients_of_an_infinite_input(shape, row):
    # an infinite input pixel of channel 3, in the last row of the image or on either side
    # of a wave's rows, makes the taps with a product of it infinite and leaves the others
    from reconnet_amd.cnn import _p, _sigs, _st

    B, H, W = shape
    rng = np.random.default_rng(row)
    a = rng.integers(-2, 3, shape + (32,)).astype(np.float64)
    d = rng.integers(1, 4, shape + (32,)).astype(np.float64)
    p = np.pad(a, ((0, 0), (1, 1), (1, 1), (0, 0)))
    want = np.stack([np.tensordot(d, p[:, t // 3:t // 3 + H, t % 3:t % 3 + W], ((0, 1, 2), (0, 1, 2)))
                     for t in range(9)])
    for t in range(9):
        if 0 <= row - (t // 3 - 1) < H:
            want[t, :, 3] = np.inf
    a[B - 1, row, 17, 3] = np.inf
    at, dt = (torch.from_numpy(v).cuda().to(torch.bfloat16) for v in (a, d))
    g, gb = torch.empty(9, 32, 32, device="cuda"), torch.empty(32, device="cuda")
    assert _sigs().rn_cnn_wgrad_mid_bias(_p(at), _p(dt), _p(g), _p(gb), B, H, W, _st()) == 0
    assert np.array_equal(g.cpu().double().numpy(), want)
