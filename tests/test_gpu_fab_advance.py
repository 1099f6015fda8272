"""Several steps of a fab level in one call against the same steps one by one:
between the steps of a call only the ghost components that the next step pulls
are filled.  The same operations on the same values, so every fab cell, ghosts
included, is equal."""
import numpy as np
import pytest

from marbles_amd import configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ncell,max_box,periodic", [
    ((12, 10, 9), 5, True),     # boxes two cells wide: one ghost row feeds both neighbours
    ((33, 17, 16), 16, True),   # a box one cell wide
    ((24, 24, 24), None, True),  # a box that is its own neighbour on every side
    ((40, 20, 24), 16, False),  # the boundary functor reads filled ghosts
])
def test_advance_equals_single_steps(engine, ncell, max_box, periodic):
    if periodic:
        cfg = configs.taylor_green(16, tau=1.0)
        cfg.update(ncell=ncell, prob_hi=tuple(float(n) for n in ncell))
    else:
        cfg = configs.channel_sphere(ncell, radius=4.0, center=(16.0, 10.0, 12.0))
    cfg["max_box"] = max_box
    a, b = (configs.build_level(cfg, layout="fab") for _ in range(2))
    a.advance(4)
    a.advance(1)
    for _ in range(5):
        b.step()
    for name in ("f", "g"):
        x, y = a.download(name), b.download(name)
        assert np.isfinite(x).all() and np.array_equal(x, y), name
    a.close()
    b.close()
