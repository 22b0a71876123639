"""The pressure operator and CR on small grids (one tile per block, one
layer of blocks) against the z-march that larger grids take."""
import numpy as np
import pytest

from tests.test_gpu_fastdiag import box_cfg

pytestmark = pytest.mark.gpu

BALL = {"center": (0.5, 0.5, 0.5), "radius": 0.17, "density": 400.0}


@pytest.fixture(scope="module")
def esf():
    import eulersf_amd
    eulersf_amd.load()
    return eulersf_amd


def pair(esf, monkeypatch, cells, precision):
    """the same box twice: as dispatched by its size, and by the march"""
    text = box_cfg(cells, [BALL] if min(cells) > 12 else [])
    out = []
    for march in (False, True):
        if march:
            monkeypatch.setenv("ESF_SPMV_LAYERS", "8")
        g = esf.CoupledIntegrator3D.from_cfg_text(text, precision)
        monkeypatch.delenv("ESF_SPMV_LAYERS", raising=False)
        g.forces()
        g.pressureDiag()
        out.append(g)
    return out


def solve(esf, g, b, x0, eps, max_it):
    A = esf._abi
    g.upload(A.F_PRESSURE_RHS, b)
    g.upload(A.F_LAMBDA, x0)
    it, ref, rr, ms, st = g.pressureSolveResident(eps, max_it)
    return it, st, rr, g.download(A.F_LAMBDA)


# one tile, one cell short of and past it; both sides of 160 tiles (the check
# beside the update), 256 (wide blocks) and 1024 (the march)
@pytest.mark.parametrize("cells", [(16, 8, 4), (15, 7, 3), (17, 9, 5), (3, 3, 50), (50, 3, 3),
                                   (64, 40, 32), (64, 40, 33), (61, 63, 32), (64, 64, 33),
                                   (128, 64, 64), (129, 64, 64)])
def test_operator_and_first_iterations_as_the_march(esf, monkeypatch, cells):
    """S x is bitwise the march's (each row summed in the reference's order).
    CR's first iterations differ by the order of the dot products alone:
    relative 2^-52 times the square root of the cells (at most 730) in each
    of alpha and beta, 12 iterations, amplified by no more than 100."""
    f, m = pair(esf, monkeypatch, cells, esf.ESF_PLAIN_FP64)
    rng = np.random.default_rng(sum(cells))
    x = rng.standard_normal(f.cells)
    np.testing.assert_array_equal(f.getMatVecMult(x), m.getMatVecMult(x))
    b = f.getMatVecMult(x)
    x0 = rng.standard_normal(f.cells)
    for max_it in (1, 2, 6, 7, 12):
        itf, stf, rrf, xf = solve(esf, f, b, x0, 1e-30, max_it)
        itm, stm, rrm, xm = solve(esf, m, b, x0, 1e-30, max_it)
        print(cells, max_it, itf, itm, stf, stm, rrf, rrm, flush=True)
        assert (itf, stf) == (itm, stm)
        assert np.linalg.norm(xf - xm) < 2e-10 * np.linalg.norm(xm)
    f.close()
    m.close()


@pytest.mark.parametrize("eps", [0.05, 2e-3])
@pytest.mark.parametrize("cells", [(17, 21, 22), (61, 41, 30), (64, 64, 33)])
def test_checked_iterate_and_last_iterations(esf, monkeypatch, cells, eps):
    """a solve stopped by its check returns the checked iterate and count,
    also where the iteration limit ends one, two or three iterations past
    it, and one short of it"""
    f, m = pair(esf, monkeypatch, cells, esf.ESF_PLAIN_FP64)
    rng = np.random.default_rng(sum(cells))
    b = f.getMatVecMult(rng.standard_normal(f.cells))
    x0 = np.zeros(f.cells)
    n, st, rr, x = solve(esf, m, b, x0, eps, 1000)
    assert st == 0
    for max_it in (1000, n + 3, n + 2, n + 1, n, n - 1):
        itf, stf, rrf, xf = solve(esf, f, b, x0, eps, max_it)
        itm, stm, rrm, xm = solve(esf, m, b, x0, eps, max_it)
        print(cells, n, max_it, itf, itm, stf, stm, rrf, rrm, flush=True)
        assert (itf, stf) == (itm, stm)
        assert np.linalg.norm(xf - xm) < 1e-8 * np.linalg.norm(xm)
    f.close()
    m.close()


def test_a_start_that_passes_is_returned_unchanged(esf, monkeypatch):
    """after a solve that iterated, the next one queues its first iterations
    before it has seen its first residual; where that passes, x is the start"""
    g, other = pair(esf, monkeypatch, (24, 21, 26), esf.ESF_MIXED)
    other.close()
    b = g.getMatVecMult(np.random.default_rng(2).standard_normal(g.cells))
    it, st, rr, x = solve(esf, g, b, np.zeros(g.cells), 1e-10, 1000)
    assert st == 0 and it > 0
    for _ in range(2):
        it2, st2, rr2, x2 = solve(esf, g, b, x, 1e-9, 1000)
        assert st2 == 0 and it2 == 0 and rr2 < 1e-9
        np.testing.assert_array_equal(x2.view(np.int64), x.view(np.int64))
    g.close()


@pytest.mark.parametrize("cells", [(16, 8, 4), (129, 64, 64)])
def test_a_refused_launch_says_why(esf, cells):
    """a runtime error found at a launch (here one left by an allocation that
    no device can grant) is named, by the small-grid operator and the march"""
    import ctypes
    g = esf.CoupledIntegrator3D.from_cfg_text(box_cfg(cells, []))
    g.forces()
    hip = ctypes.CDLL("libamdhip64.so.7")
    p = ctypes.c_void_p()
    assert hip.hipMalloc(ctypes.byref(p), ctypes.c_size_t(1 << 60)) != 0
    with pytest.raises(esf._abi.EsfError, match="launch: out of memory"):
        g.getMatVecMult(np.zeros(g.cells))
    assert not g.getMatVecMult(np.zeros(g.cells)).any()
    g.close()
