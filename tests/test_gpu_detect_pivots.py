"""The detector on singular and infinite channels: a pivot of zero has an
infinite reciprocal and an infinite pivot a zero one, as by division, and what
follows is fp32 arithmetic.  One layer against the formula in numpy; two layers
where the second pivot cancels to zero."""
import numpy as np
import pytest

from puschrx import ops
from puschrx import profiles as P

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _detect(rank, h, y, no):
    """h [nr, rank, n], y [nr, n], no [4] (real, fp16) on the first n REs -> xhat re, im and no_eff [rank, n]."""
    cfg = P.Profile(name="t", rx=4, rank=rank, num_rb=6, fft=128, qm=4, padded_subcarriers=128).config()
    g = ops.Geometry(cfg)
    n = y.shape[1]
    hg = np.zeros((g.nr, 16, g.n_re), np.float16)
    yg = np.zeros((g.nr, g.n_re), np.float16)
    hg[:, :rank, :n], yg[:, :n] = h, y
    dev = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    packed = ops.detect_io_pack(cfg, dev(yg), dev(np.zeros_like(yg)), dev(hg), dev(np.zeros_like(hg)),
                                dev(np.asarray(no, np.float16)))
    out = ops.detect_lmmse(cfg, *packed)
    torch.cuda.synchronize()
    return [o.cpu().numpy().reshape(-1, g.n_re)[:rank, :n] for o in out]


@pytest.mark.parametrize("no", [0.0, 2.0 ** -24, 0.25])
def test_one_layer(gpu_stream, no):
    inf = np.inf
    col = np.array([0.0, inf, -inf, 2.0 ** -24, 65504.0, 1.0, np.nan], np.float16)
    h0, y0 = (a.reshape(-1) for a in np.meshgrid(col, np.array([0.0, 1.0, -2.0, inf], np.float16)))
    h, y = np.zeros((4, 1, h0.size), np.float16), np.zeros((4, h0.size), np.float16)
    h[0, 0], y[0] = h0, y0
    xr, _, ne = _detect(1, h, y, [no] * 4)
    f = np.float32
    with np.errstate(all="ignore"):
        inv = f(1) / (h0.astype(f) ** 2 + f(no))
        d = np.fmax(f(1) - f(no) * inv, f(1e-3))
        want_x = (h0.astype(f) * y0.astype(f) * inv / d).astype(np.float16)
        want_n = ((f(1) - d) / d).astype(np.float16)
    for got, want in ((xr[0], want_x), (ne[0], want_n)):
        special = ~np.isfinite(want)
        np.testing.assert_array_equal(np.where(special, got, 0), np.where(special, want, 0))
        # Finite values: two roundings of 2^-24 each against this formula's, then to fp16.
        np.testing.assert_allclose(got[~special].astype(f), want[~special].astype(f), rtol=2.0 ** -10, atol=2.0 ** -24)


def test_two_layers_second_pivot_zero(gpu_stream):
    """h1 = h0 + 2^-13 e1: |h1|^2 rounds to 1 in fp32, so the second pivot is
    0 without noise and its layer's estimate infinite by the sign of y1."""
    y1 = np.array([1.0, -1.0, 3.0], np.float16)
    h, y = np.zeros((4, 2, 3), np.float16), np.zeros((4, 3), np.float16)
    h[0], h[1, 1], y[1] = 1.0, 2.0 ** -13, y1
    xr, _, ne = _detect(2, h, y, [0.0] * 4)
    assert np.array_equal(xr[1], np.where(y1 > 0, np.inf, -np.inf))
    assert np.all(ne == np.float16(999.0))
