"""The Stockham passes with register ends (first and last stage without LDS)
against the passes that stage every value, which a tile of three pairs selects:
the same arithmetic, so the same bits, on lengths whose last stage is each of
the radices 8, 4, 2, 3 and 5, at the shortest lengths that take the form and
on both launch classes (one field, the strided batch)."""
import numpy as np
import pytest

from ib_parallel_amd import abi, decks
from ib_parallel_amd.abi import make_params

pytestmark = pytest.mark.gpu


def _run(monkeypatch, shape, tiles):
    from ib_parallel_amd import GpuSim
    monkeypatch.setenv("IB_DST_FORM", "fft")
    monkeypatch.delenv("IB_DST_TILES", raising=False)
    if tiles:
        monkeypatch.setenv("IB_DST_TILES", tiles)
    m, n = shape
    p = make_params(m, n, 2, 0.001, 100.0, 4.0, 1.0, 2.0 * n / m, num_stat=1)
    g = GpuSim(p, [decks.cylinder_body(24, radius=0.15)])
    a = np.random.default_rng(7).standard_normal(g.P)
    d = g.dst2d(a)
    for _ in range(3):
        assert g.advance().status == abi.IB_OK
    out = [d, g.ctci(a), g.ainv(a), g.schur_matrix(), g.body()["f"]]
    out += [g.level(k)[q] for k in (1, 2) for q in ("omega", "s")]
    g.close()
    return a, out


# transform lengths 2m, 2n: 640 = 8 8 2 5, 400 = 8 2 5 5; 768 = 8 8 4 3, 512 = 8 8 8;
# 800 = 8 4 5 5; 1024 = 8 8 8 2, 648 = 8 3 3 3 3; 2048 = 8 8 8 4
@pytest.mark.parametrize("shape", ((320, 200), (384, 256), (400, 400), (512, 324), (1024, 200)))
def test_register_ends_keep_the_bits(monkeypatch, shape):
    a, want = _run(monkeypatch, shape, "3,3")
    for tiles in ("1,1", "4,4", None):
        _, got = _run(monkeypatch, shape, tiles)
        for w, x in zip(want, got):
            assert np.array_equal(w, x), (shape, tiles)
    # and the plain transform against the sine sums: 2(M-1) terms of eps each at most
    m, n = shape
    S = [np.sin(np.pi * np.outer(np.arange(1, q), np.arange(1, q)) / q) for q in (n, m)]
    ref = 4 * S[0] @ a.reshape(n - 1, m - 1) @ S[1]
    assert np.abs(want[0].reshape(ref.shape) - ref).max() <= 2e-13 * np.abs(ref).max()
