"""The sweeps' 8 x 8-row tiles at their edges, against the oracle bit for bit:
boxes whose rows end on a tile, one past it and inside the first, flat and
long ones, and two calls in a row through one context's hand-over buffer."""
import numpy as np
import pytest

from oracle import oracle as O
from tests._scenes import ball_cfg

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def esf():
    import eulersf_amd
    eulersf_amd.load()
    return eulersf_amd


def context(esf, nodes):
    text = ball_cfg(63)
    for axis, n in zip("xyz", nodes):
        text = text.replace("%sRes = 64" % axis, "%sRes = %d" % (axis, n))
    return esf.CoupledIntegrator3D.from_cfg_text(text.replace("number of solids = 1", "number of solids = 0"))


def blobs(nodes, seed):
    rng = np.random.default_rng(seed)
    m = np.zeros(nodes[::-1])
    for _ in range(2):
        c = [rng.integers(0, n) for n in nodes[::-1]]
        m[tuple(slice(max(a - 1, 0), a + 2) for a in c)] = rng.uniform(0.5, 2.0)
    return m


# the box is the whole grid (20 extrapolation cells): a sweep of phi has
# n - 1 rows per axis, a field pass n - 2
@pytest.mark.parametrize("nodes", [(4, 4, 4), (9, 9, 9), (10, 10, 10), (11, 17, 18), (18, 10, 19),
                                   (40, 5, 26), (5, 34, 9), (33, 25, 41)])
def test_sweeps_bitwise_at_tile_edges(esf, nodes):
    g = context(esf, nodes)
    for seed in (1, 2):
        m = blobs(nodes, seed)
        phi, box, tight = g.computeSDF(m)
        phi_o, box_o, tight_o = O.compute_sdf(m, 5, 20)
        assert list(box) == list(box_o) and list(tight) == list(tight_o)
        assert np.array_equal(phi.view(np.int64), phi_o.view(np.int64))
        phi_n, _, _ = g.computeSDFNoAlloc(m)
        assert np.array_equal(phi_n.view(np.int64), phi_o.view(np.int64))
        f = np.random.default_rng(seed).normal(size=m.shape + (3,))
        out, out_o = g.extendVectorField(box, m, phi, f), O.extend_vector_field(m, phi_o, box_o, f)
        assert np.array_equal(out.view(np.int64), out_o.view(np.int64))
    g.close()


def test_a_field_with_infinities_passes_through(esf):
    """hand-over words carry any bits: an infinite and a NaN component"""
    nodes = (20, 20, 20)
    g = context(esf, nodes)
    m = blobs(nodes, 3)
    phi, box, _ = g.computeSDF(m)
    f = np.random.default_rng(3).normal(size=m.shape + (3,))
    f[m > 0, 1] = np.inf
    f[m > 0, 2] = np.nan
    out, out_o = g.extendVectorField(box, m, phi, f), O.extend_vector_field(m, phi, box, f)
    np.testing.assert_array_equal(out, out_o)
    assert np.isinf(out[..., 1]).any() and np.isnan(out[..., 2]).any()
    g.close()
