"""Macroscopic fields and vorticity where the read-outs' blocks of 256
consecutive cells and the rows do not line up (rows of less than, about and
more than 256 cells, a nearly empty last block), every storage: density and
velocity against the sums over the downloaded populations, vorticity against
the oracle (FP64).  Tolerances: a sum of 27 values of order 1e-1 in FP64
differs by 27 x 1e-16 at most, 1e-14; vorticity 1e-12 of the largest."""
import numpy as np
import pytest
import torch

from marbles_amd import configs
from marbles_amd.stencil import velocity_density

pytestmark = pytest.mark.gpu

SIZES = [(37, 19, 13), (255, 10, 9), (257, 9, 10), (300, 12, 11)]


def _cfg(n):
    return configs.channel_sphere(n, radius=2.5, center=(12.0, n[1] / 2, n[2] / 2))


@pytest.mark.parametrize("storage", ["f64", "f32s", "f16s"])
@pytest.mark.parametrize("n", SIZES)
def test_macro_fields_at_ragged_rows(engine, n, storage):
    E = configs.build_level(_cfg(n), layout="compact", storage=storage)
    E.advance(5)
    out = torch.full((5, n[2], n[1], n[0]), -7.0, dtype=torch.float64, device="cuda")
    E.macro_fields(out)
    torch.cuda.synchronize()
    got, f, fluid = out.cpu().numpy(), E.valid("f"), E.valid("is_fluid")[0] == 1
    E.close()
    vel, rho = velocity_density(np.where(fluid, f, 0.0))
    assert 0 < fluid.sum() < fluid.size
    for a, b in zip(got[:4], [rho] + vel):
        assert np.abs(a - b).max() <= 1e-14
    assert (got[4][fluid] > 0).all() and (got[:, ~fluid] == 0).all()


@pytest.mark.parametrize("n", SIZES)
def test_vorticity_at_ragged_rows(oracle, engine, n):
    from oracle.pyoracle import build_oracle_level

    cfg = _cfg(n)
    O = build_oracle_level(cfg)
    O.evolve(5)
    ref = O.vorticity()
    E = configs.build_level(cfg, layout="compact")
    E.advance(5)
    out = torch.empty(4 * int(np.prod(n)), dtype=torch.float64, device="cuda")
    E.vorticity(out)
    torch.cuda.synchronize()
    got = out.cpu().numpy().reshape(ref.shape)
    E.close()
    assert np.abs(got - ref).max() <= 1e-12 * np.abs(ref[3]).max()
