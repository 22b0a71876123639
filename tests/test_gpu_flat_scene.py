"""A cfg whose smoke carpet is thicker than the box is high."""
import numpy as np
import pytest

from eulersf_amd.cfg import scene_cfg

pytestmark = pytest.mark.gpu


def test_carpet_thicker_than_the_box_ends_at_its_top():
    import eulersf_amd as esf
    text = scene_cfg(32, []).replace("yRes = 33", "yRes = 4")  # 9 layers of carpet, 4 of nodes
    g = esf.CoupledIntegrator3D.from_cfg_text(text)
    smoke = g.download(esf._abi.F_INTENSITY).reshape(33, 4, 33)
    expect = np.zeros_like(smoke)
    expect[1:-1, 1:, 1:-1] = np.float32(0.8)
    np.testing.assert_array_equal(smoke, expect)
    g.close()
