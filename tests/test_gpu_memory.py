"""Steps whose allocations fail: the call reports it, and the engine works
again once there is memory."""
import numpy as np
import pytest

from ziran2019_amd import scenes
from ziran2019_amd.engine import MpmEngine, ZrError
from _device_memory import device_memory_held
from _helpers import make_pair

pytestmark = pytest.mark.gpu


def _spread(n):
    """n particles, most of them in a page of their own."""
    rng = np.random.default_rng(5)
    cube = scenes.cube_scene_small(seed=3, ncells=4)
    s = {k: np.resize(cube[k], (n,) + cube[k].shape[1:]) for k in ("V", "C", "F", "mass", "vol", "mu", "lam")}
    return dict(s, X=0.05 + 0.85 * rng.random((n, 3)), dx=1.0 / 256)


def _same(a, b):
    for k in a:
        assert np.array_equal(a[k], b[k]), k


def test_a_sort_that_finds_no_memory_leaves_nothing_behind():
    """The first sort of many groups allocates the cells' table (38 MB here)
    after the pages have been counted."""
    n = 300000
    s = _spread(n)
    ref = MpmEngine(dx=s["dx"])
    ref.upload(s)
    for _ in range(2):
        ref.advanceOneTimeStep(1e-5)
    want = ref.download()
    ref.close()
    small = {k: (v[:50000] if isinstance(v, np.ndarray) else v) for k, v in s.items()}
    eng = MpmEngine(dx=s["dx"])
    eng.upload(small)
    eng.advanceOneTimeStep(1e-5)
    eng.upload(s)
    with device_memory_held(eng.L, 8 << 20):
        with pytest.raises(ZrError, match="memory"):
            eng.advanceOneTimeStep(1e-5)
    for _ in range(2):
        eng.advanceOneTimeStep(1e-5)
    _same(eng.download(), want)
    eng.close()


def test_a_grid_that_finds_no_memory_is_not_used():
    """The grid's arrays are freed for larger ones (59 MB the smallest), which
    are not to be had: the next step does not take the old capacity for
    granted, nor an upload of as many particles the arrays of one that failed."""
    cube = scenes.cube_scene_small(seed=3, ncells=8, lo_cell=80, dx=1.0 / 256)
    eng, _ = make_pair(cube)
    eng.advanceOneTimeStep(1e-4)
    first = eng.download()
    eng.advanceOneTimeStep(1e-4)
    want = eng.download()
    eng.upload(_spread(50000))
    with device_memory_held(eng.L, 16 << 20):
        with pytest.raises(ZrError, match="memory"):
            eng.advanceOneTimeStep(1e-6)
    eng.upload(dict(cube, **first))
    eng.advanceOneTimeStep(1e-4)
    _same(eng.download(), want)
    with device_memory_held(eng.L, 8 << 20):
        for _ in range(2):
            with pytest.raises(ZrError, match="memory"):
                eng.upload(_spread(300000))
            with pytest.raises(ZrError, match="no particles"):
                eng.advanceOneTimeStep(1e-4)
    eng.upload(dict(cube, **first))
    eng.advanceOneTimeStep(1e-4)
    _same(eng.download(), want)
    eng.close()


def _shuffled(n):
    s = scenes.cube_scene(dx=1.0 / 128, lo_cell=40, ncells=34)
    p = np.random.default_rng(6).permutation(len(s["mass"]))[:n]
    return {k: (np.ascontiguousarray(v[p]) if isinstance(v, np.ndarray) else v) for k, v in s.items()}


def test_particles_stay_where_their_second_copy_finds_no_memory():
    """A shuffled set is moved at its second step where there is memory for a
    second copy (71 MB)."""
    s = _shuffled(300000)
    outs = []
    for left in (None, 8 << 20):
        eng, _ = make_pair(s, colliders=s["colliders"])
        eng.advanceOneTimeStep(1e-4)
        if left is None:
            for _ in range(3):
                eng.advanceOneTimeStep(1e-4)
        else:
            with device_memory_held(eng.L, left):
                for _ in range(3):
                    eng.advanceOneTimeStep(1e-4)
        outs.append(eng.download())
        eng.close()
    _same(*outs)


def test_second_copies_are_given_back():
    """A call that needs memory takes that of the second copies (71 MB, the
    checkpoint 58 MB); without them the caller's order is restored row by row."""
    s = _shuffled(300000)
    ref, _ = make_pair(s, colliders=s["colliders"])
    eng, _ = make_pair(s, colliders=s["colliders"])
    for e in (ref, eng):
        for _ in range(3):
            e.advanceOneTimeStep(1e-4)
    want = ref.download()
    ref.advanceOneTimeStep(1e-4)
    after = ref.download()
    ref.sortParticlesAndPolluteGrid()
    order = ref.dump("order")
    ref.close()
    with device_memory_held(eng.L, 8 << 20):
        eng.checkpoint_save(0)
        eng.sortParticlesAndPolluteGrid()
        eng.dump("order")  # in the caller's order from here on
        _same(eng.download(), want)
        eng.advanceOneTimeStep(1e-4)
        _same(eng.download(), after)
        eng.sortParticlesAndPolluteGrid()
        assert np.array_equal(eng.dump("order"), order)
        eng.checkpoint_restore(0)
        _same(eng.download(), want)
    eng.close()


def test_an_engine_that_finds_no_memory_fails_alone():
    """The page tables of an extent of 2^12 nodes take 34 GB; another engine's
    next step does not report their failure."""
    cube = scenes.cube_scene_small(seed=3, ncells=4)
    eng, _ = make_pair(cube)
    eng.advanceOneTimeStep(1e-4)
    with device_memory_held(eng.L, 64 << 20):
        with pytest.raises(ZrError):
            MpmEngine(dx=cube["dx"], grid_log2=12)
        eng.advanceOneTimeStep(1e-4)
    eng.close()
