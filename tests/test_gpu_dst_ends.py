"""The Stockham passes with register ends (first and last stage without LDS)
against the passes that stage every value: the same arithmetic, so the same
bits, on lengths whose last stage is each of the radices 8, 4, 2, 3 and 5 in
rows and in columns, from the shortest plans on, with one, two and four pairs
per workgroup and on both launch classes (one field, the strided batch).
IB_DST_FORM=fft:staged keeps the staged passes whatever the tile;
IB_DST_FORM=fft:ends fails where a pass would not take register ends."""
import numpy as np
import pytest

from ib_parallel_amd import abi, decks
from ib_parallel_amd.abi import make_params
from ib_parallel_amd.sim import IBError

pytestmark = pytest.mark.gpu


def _sim(monkeypatch, shape, form, tiles):
    from ib_parallel_amd import GpuSim
    monkeypatch.setenv("IB_DST_FORM", form)
    monkeypatch.delenv("IB_DST_TILES", raising=False)
    if tiles:
        monkeypatch.setenv("IB_DST_TILES", tiles)
    m, n = shape
    p = make_params(m, n, 2, 0.001, 100.0, 4.0, 1.0, 2.0 * n / m, num_stat=1)
    return GpuSim(p, [decks.cylinder_body(24 if m >= 128 else 6, radius=0.15)])


def _run(monkeypatch, shape, form, tiles):
    g = _sim(monkeypatch, shape, form, tiles)
    a = np.random.default_rng(7).standard_normal(g.P)
    d = g.dst2d(a)
    for _ in range(3):
        assert g.advance().status == abi.IB_OK
    out = [d, g.ctci(a), g.ainv(a), g.schur_matrix(), g.body()["f"]]
    out += [g.level(k)[q] for k in (1, 2) for q in ("omega", "s")]
    g.close()
    return a, out


# transform lengths 2m, 2n: 64 = 8 8, 32 = 8 4; 128 = 8 8 2; 256 = 8 8 4, 192 = 8 8 3;
# 640 = 8 8 2 5, 400 = 8 2 5 5; 768 = 8 8 4 3, 512 = 8 8 8; 800 = 8 4 5 5;
# 1024 = 8 8 8 2, 648 = 8 3 3 3 3; 2048 = 8 8 8 4
@pytest.mark.parametrize("shape", ((32, 16), (64, 64), (128, 96), (96, 128), (320, 200), (384, 256), (400, 400),
                                   (512, 324), (512, 512), (1024, 200), (320, 1024)))
def test_register_ends_keep_the_bits(monkeypatch, shape):
    a, want = _run(monkeypatch, shape, "fft:staged", "1,1")
    for form, tiles in (("fft:ends", "1,1"), ("fft:ends", "2,2"), ("fft:ends", "4,4"), ("fft", None)):
        _, got = _run(monkeypatch, shape, form, tiles)
        for w, x in zip(want, got):
            assert np.array_equal(w, x), (shape, form, tiles)
    # and the plain transform against the sine sums: 2(M-1) terms of eps each at most
    m, n = shape
    S = [np.sin(np.pi * np.outer(np.arange(1, q), np.arange(1, q)) / q) for q in (n, m)]
    ref = 4 * S[0] @ a.reshape(n - 1, m - 1) @ S[1]
    assert np.abs(want[0].reshape(ref.shape) - ref).max() <= 2e-13 * np.abs(ref).max()


def test_register_ends_are_not_replaced_silently(monkeypatch):
    """A tile of three pairs and a radix of 7 (2 x 56 = 8 2 7) have no pass with
    register ends: asked for by name it is an error, else the staged pass."""
    with pytest.raises(IBError, match="register ends"):
        _run(monkeypatch, (128, 64), "fft:ends", "3,3")
    with pytest.raises(IBError, match="register ends"):
        _run(monkeypatch, (56, 64), "fft:ends", "1,1")
    for shape, tiles in (((128, 64), "3,3"), ((56, 64), "1,1")):
        _, want = _run(monkeypatch, shape, "fft:staged", "1,1")
        _, got = _run(monkeypatch, shape, "fft", tiles)
        assert all(np.array_equal(w, x) for w, x in zip(want, got))
