"""The cooperative GMRES solve (gmres_form 2 up to nf = 256, 0/4 up to nf =
1024) at the edges of its layout: the last workgroup with few rows, a number of
workgroups that is not a power of two, the change from direct sums of the
partial coefficients to published ones, restarts, basis vectors past the LDS,
an initial guess that already satisfies the tolerance."""
import ctypes as C

import numpy as np
import pytest

from conftest import rel
from ib_parallel_amd import abi, decks
from ib_parallel_amd.sim import IBError

pytestmark = pytest.mark.gpu


def _circle(npts, **kw):
    m = 4 * max(12, round(npts / np.pi))  # points one cell apart
    p, _ = decks.cylinder_case(m=m, n=m, mgridlev=1, npts=npts, tol=1e-11, **kw)
    return p, [decks.cylinder_body(npts)]


def _solve(mk, form, x0=0.9, seed=5):
    from ib_parallel_amd import GpuSim
    g = GpuSim(*mk(form))
    S = g.schur_matrix()
    xt = np.random.default_rng(seed).standard_normal(g.nf)
    b = S @ xt
    x, its = g.gmres(b, x0=x0 * xt, allow_noconv=True)
    info, nf = g.gmres_info(), g.nf
    g.close()
    return x, its, np.linalg.norm(S @ x - b) / np.linalg.norm(b), info, nf


# (points, gmres_form, restart, workgroups expected): 42 entries as 2 x 21
# rows, 48 as 8 x 6, 256 as 4 x 64 (and 8 x 32 where the basis needs the LDS),
# 260 in 16 workgroups of 17 (the last one 5 rows), 520 in 31 of 17 (the last
# one 10), 1024 in 32 of 32
@pytest.mark.parametrize("npts, form, restart, groups", [(21, 2, 400, 2), (24, 4, 400, 8), (128, 2, 250, 4), (128, 2, 400, 8),
                                                         (130, 0, 400, 16), (260, 0, 400, 31), (512, 0, 400, 32)])
def test_cooperative_gmres_at_layout_edges(npts, form, restart, groups):
    """Against the per-stage kernels (gmres_form 3) on the same matrix: the
    same iteration with its sums in another order, so the iteration counts
    agree within one, and both residuals meet the tolerance (the recurrence's
    estimate and the true residual part by rounding times the condition number,
    below 1e5 for points one cell apart)."""
    mk = lambda f: _circle(npts, gmres_restart=restart, gmres_form=f)
    x, its, r, info, nf = _solve(mk, form)
    x3, its3, r3, info3, _ = _solve(mk, 3)
    assert nf == 2 * npts and info[0] == (2 if form == 2 else 3) and info[1] == groups and info3[0] == 0, (info, info3)
    assert abs(its - its3) <= 1, (its, its3)
    assert r < 1e-10 and r3 < 1e-10, (r, r3)
    assert rel(x, x3) < 1e-7


@pytest.mark.parametrize("npts, form", [(21, 2), (130, 0)])
@pytest.mark.parametrize("restart", (1, 2, 7))
def test_cooperative_gmres_restarts(npts, form, restart):
    """Short cycles, so that the exchange buffers are cleared and used again:
    40 iterations from the same guess (more than the solve needs is not
    allowed: gmres_max_it) leave the solution of the per-stage kernels to
    rounding, which a cycle amplifies by little."""
    mk = lambda f: _circle(npts, gmres_restart=restart, gmres_max_it=40, gmres_form=f)
    x, its, r, info, _ = _solve(mk, form)
    x3, its3, r3, _, _ = _solve(mk, 3)
    assert info[0] in (2, 3) and its == its3 == 40, (its, its3)
    assert abs(r - r3) < 1e-9 * max(r3, 1e-3) and rel(x, x3) < 1e-9


def test_cooperative_gmres_basis_past_the_lds(monkeypatch):
    """Basis vectors past the LDS share keep their arithmetic: the same bits,
    over restarts too."""
    mk = lambda f: _circle(130, gmres_restart=90, gmres_form=f)
    x, its, r, info, _ = _solve(mk, 0)
    monkeypatch.setenv("IB_COOPW_LDS_VECTORS", "5")
    y, its5, _, info5, _ = _solve(mk, 0)
    assert info[0] == info5[0] == 3 and its == its5 and its > 5
    assert np.array_equal(x, y)


def test_cooperative_gmres_from_the_solution():
    """A guess that meets the tolerance ends before the first step and stays."""
    mk = lambda f: _circle(130, gmres_restart=30, gmres_form=f)
    x, its, r, info, _ = _solve(mk, 0, x0=1.0)
    assert info[0] == 3 and its == 0 and r < 1e-11


@pytest.mark.parametrize("npts, form, groups", [(21, 2, 2), (130, 0, 16)])
@pytest.mark.parametrize("exchange", ("1", "0"))
def test_a_workgroup_that_gives_up_fails_the_solve(monkeypatch, npts, form, groups, exchange):
    """A workgroup whose last wait times out leaves without its rows of the
    solution: the solve reports the time-out, whichever workgroup it is and
    although all the others finish, and the next solve on the handle is whole."""
    from ib_parallel_amd import GpuSim
    monkeypatch.setenv("IB_GMRES_L2_EXCHANGE", exchange)
    g = GpuSim(*_circle(npts, gmres_restart=400, gmres_form=form))
    assert g.gmres_info()[1] == groups
    b = g.schur_matrix() @ np.random.default_rng(5).standard_normal(g.nf)
    want = g.gmres(b)
    for rank in (0, 1, groups - 1):
        monkeypatch.setenv("IB_GMRES_FAIL_RANK", str(rank))
        with pytest.raises(IBError) as e:
            g.gmres(b)
        assert e.value.code == abi.IB_E_HIP and "timed out" in str(e.value), (rank, str(e.value))
        monkeypatch.delenv("IB_GMRES_FAIL_RANK")
        x, its = g.gmres(b)
        assert its == want[1] and np.array_equal(x, want[0])
    g.close()


def test_workspace_of_the_small_form_is_what_it_lays_out():
    """nf = 200 at restart 1000, 16 workgroups: one Hessenberg matrix (8 MB) and
    the exchange buffers (3 x 1001 x 16 values), not a matrix per workgroup.
    Against a handle of the one-workgroup solve, which keeps no such workspace;
    4 MB for the allocator's granularity."""
    from ib_parallel_amd import GpuSim, library
    hip = library()
    hip.hipMemGetInfo.argtypes = [C.POINTER(C.c_size_t), C.POINTER(C.c_size_t)]

    def taken(form, groups):
        free, total = [C.c_size_t() for _ in range(2)], C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(free[0]), C.byref(total)) == 0
        g = GpuSim(*_circle(100, gmres_restart=1000, gmres_form=form))
        assert hip.hipMemGetInfo(C.byref(free[1]), C.byref(total)) == 0
        assert g.gmres_info()[:2] == (form, groups)
        return g, free[0].value - free[1].value

    for form, groups in ((1, 1), (2, 16)):  # what the runtime takes once
        taken(form, groups)[0].close()
    one, base = taken(1, 1)
    two, mem = taken(2, 16)
    one.close()
    two.close()
    words = 1000 * 1001 + 3 * 1001 * 16 + 4 * 1001 + 4 * 200 + 3 * 1000 + 2 * 16 + 40
    assert mem - base < 8 * words + (4 << 20), (mem, base)
