"""Downloads past the size from which several threads carry them: whole and
partial chunks, more callers at once than there are sets of slots, and slots
taken anew after the last context went."""
import threading

import numpy as np
import pytest

from eulersf_amd.cfg import scene_cfg

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def esf():
    import eulersf_amd
    eulersf_amd.load()
    return eulersf_amd


def context(esf, n):
    return esf.CoupledIntegrator3D.from_cfg_text(scene_cfg(n, []))


# velocity of 2.82, 3.18 (just past the threshold of 3 MiB), 6.59 and 13.2 MB
@pytest.mark.parametrize("n", [48, 50, 64, 81])
def test_download_returns_what_was_uploaded(esf, n):
    g = context(esf, n)
    v = np.random.default_rng(n).standard_normal(3 * g.nodes)
    g.upload(esf._abi.F_VELOCITY, v)
    np.testing.assert_array_equal(g.download(esf._abi.F_VELOCITY), v)
    g.close()


def test_more_callers_than_slots(esf):
    scenes = [context(esf, 64) for _ in range(6)]
    want = [np.random.default_rng(k).standard_normal(3 * g.nodes) for k, g in enumerate(scenes)]
    for g, v in zip(scenes, want):
        g.upload(esf._abi.F_VELOCITY, v)
    bad = []

    def read(k):
        for _ in range(4):
            if not np.array_equal(scenes[k].download(esf._abi.F_VELOCITY), want[k]):
                bad.append(k)

    team = [threading.Thread(target=read, args=(k,)) for k in range(len(scenes))]
    for t in team:
        t.start()
    for t in team:
        t.join()
    assert not bad
    for g in scenes:
        g.close()


@pytest.mark.parametrize("n", [50, 64, 81])
def test_downloads_once_slots_are_pinned(esf, n):
    """past 48 MiB of large copies they go through the slots: whole and partial
    chunks, and again in a context made after the slots went with the last"""
    for turn in range(2):
        g = context(esf, n)
        v = np.random.default_rng(10 * n + turn).standard_normal(3 * g.nodes)
        g.upload(esf._abi.F_VELOCITY, v)
        for _ in range(48 * 2 ** 20 // v.nbytes + 3):
            np.testing.assert_array_equal(g.download(esf._abi.F_VELOCITY), v)
        g.close()
