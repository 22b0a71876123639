"""The solid displacement's advection, at each number of layers that a tile
marches, and the solid operator over more solids than one small table holds."""
import numpy as np
import pytest

from tests._scenes import ball_cfg, rel_err
from eulersf_amd.cfg import scene_cfg
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def esf():
    import eulersf_amd
    eulersf_amd.load()
    return eulersf_amd


# 2, 4 and 8 layers per tile, the last tile partial in x, y and z
@pytest.mark.parametrize("n", [16, 80, 96])
def test_displacement_advection_at_each_march(esf, n):
    """random u and velocity, departure points up to four cells away: inside
    the tile's window and far from it.  Error: the departure point's cell
    coordinate rounds by about n 2^-52, times differences of at most 10
    between corners, plus some 60 roundings of values of at most 6: below
    6e-13 for n <= 96."""
    A = esf._abi
    text = ball_cfg(n, velocity=(0.3, -1.0, 0.2))
    g = esf.CoupledIntegrator3D.from_cfg_text(text)
    o = O.OracleScene.from_cfg_text(text)
    dt = g.CFL(1.8)
    o.L.orc_cfl(o.h, 1.8)
    rng = np.random.default_rng(n)
    nodes = (n + 1) ** 3
    u = rng.uniform(-1, 1, 3 * nodes)
    v = rng.uniform(-1, 1, (nodes, 3)) * rng.choice([0.5, 4.0], (nodes, 1)) / (n * dt)
    for gf, of, val in ((A.S_U, O.S_U, u), (A.S_VELOCITY, O.S_VELOCITY, v.reshape(-1))):
        g.upload(gf, val, 0)
        o.set_field(of, val, 0)
    g.solidFinalize()
    o.L.orc_solid_finalize(o.h)
    np.testing.assert_allclose(g.download(A.S_U, 0), o.field(O.S_U, 0), rtol=0, atol=1e-12)
    g.close()
    o.close()


@pytest.mark.parametrize("count", [3, 4, 6])
def test_solid_operator_over_few_and_many_solids(esf, count):
    """A x of the solid system with as many solids as the small table of the
    cell pass holds and with more, against the oracle's; 64-bit sums of at
    most 8 cells x 24 terms per row"""
    at = [(0.25 + 0.25 * (i % 3), 0.3 + 0.35 * (i // 3), 0.5) for i in range(count)]
    spheres = [{"center": c, "radius": 0.09, "density": 500.0 + 200.0 * i}
               for i, c in enumerate(at)]
    text = scene_cfg(28, spheres)
    g = esf.CoupledIntegrator3D.from_cfg_text(text)
    o = O.OracleScene.from_cfg_text(text)
    g.CFL(1.8)
    o.L.orc_cfl(o.h, 1.8)
    g.forces()
    o.L.orc_forces(o.h)
    o.L.orc_assemble(o.h)
    assert g.num_solid_nodes() == o.num_solid_nodes()
    x = np.random.default_rng(count).standard_normal(3 * g.num_solid_nodes())
    assert rel_err(g.solidApply(x), o.solid_apply(x)) < 1e-12
    g.close()
    o.close()
