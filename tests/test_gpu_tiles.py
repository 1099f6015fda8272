"""The two-pass step on tiles of consecutive cells (both passes in one launch
on large FP64 levels) against the same step on blocks of rows, bit for bit:
the passes do the same arithmetic on the same pulled values, so the tolerance
is zero."""
import numpy as np
import pytest

from marbles_amd import configs

pytestmark = pytest.mark.gpu

# (storage, tile variant, row-block variant of the same arithmetic)
PAIRS = {
    "f64": ("k_qpass_x256+k_collide_x256", "k_qpass+k_collide"),
    "f32s": ("k_qpass_x256+k_collide_f32_x256", "k_qpass_y2+k_collide_f32"),
    "f32s_fp64": ("k_qpass_x256+k_collide_x256", "k_qpass+k_collide"),
    "f16s_fp64": ("k_qpass_x256+k_collide_x256", "k_qpass+k_collide"),
}


def _levels(cfg, storage, names):
    out = []
    for name in names:
        E = configs.build_level(cfg, layout="compact", storage=storage)
        E.set_hot_kernel(name)
        out.append(E)
    return out


# planes of one cell less, exactly and one cell more than a tile (and than the
# 128-cell tile of FP32 storage), rows longer than a tile, single rows and
# planes; the last three lie around the size from which an FP64 level takes
# both passes in one launch (2^18 cells), the work list longer than a plane
SHAPES = [(17, 15, 5), (16, 16, 4), (257, 1, 3), (129, 1, 2), (300, 3, 1), (5, 3, 40), (63, 64, 65), (64, 64, 64),
          (301, 30, 30)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("storage", sorted(PAIRS))
def test_tile_step_equals_row_blocks_bitwise(engine, shape, storage):
    cfg = configs.taylor_green(16, tau=1.0)
    cfg.update(ncell=shape, prob_hi=tuple(float(n) for n in shape))
    a, b = _levels(cfg, storage.split("_")[0], PAIRS[storage])
    for _ in range(3):
        a.advance(1)
        b.advance(1)
    for name in ("f", "g"):
        x, y = a.valid(name), b.valid(name)
        assert np.isfinite(x).all() and np.array_equal(x, y), (shape, storage, name)
    a.close()
    b.close()


@pytest.mark.parametrize("storage", ["f64", "f32s"])
@pytest.mark.parametrize("case", ["sphere", "duct", "parabolic_y", "pressure", "sphere_large", "duct_large"])
def test_tile_step_boundaries_bitwise(engine, storage, case):
    """Solid cells, walls, profile inlets (on x-lo, the specialised lookup,
    and on y-lo) and pressure faces in tiles that straddle rows."""
    if case == "sphere":
        cfg = configs.channel_sphere((45, 23, 21), radius=5.0, center=(16.0, 11.0, 10.0))
    elif case == "sphere_large":
        cfg = configs.channel_sphere((131, 47, 45), radius=9.0, center=(40.0, 23.0, 22.0))
    elif case == "duct":
        cfg = configs.channel_profile((37, 19, 18))
    elif case == "duct_large":
        cfg = configs.channel_profile((131, 47, 45))
    elif case == "parabolic_y":
        cfg = configs.cylinder_deck("single_cylinder", scale=6)
    else:
        cfg = configs.pressure_case("walled")
    names = PAIRS[storage] if case != "pressure" else PAIRS["f32s_fp64"]
    a, b = _levels(cfg, storage, names)
    for _ in range(4):
        a.advance(1)
        b.advance(1)
    for name in ("f", "g"):
        assert np.array_equal(a.valid(name), b.valid(name)), (case, storage, name)
    a.close()
    b.close()


def test_one_launch_step_replayed_from_a_graph(engine):
    """The work list's counter carries over from launch to launch: one captured
    step, replayed with eager steps between the replays, equals eager steps."""
    import torch

    cfg = configs.channel_sphere((131, 47, 45), radius=9.0, center=(40.0, 23.0, 22.0))
    a, b = _levels(cfg, "f64", (PAIRS["f64"][0],) * 2)
    s = torch.cuda.Stream()
    a.advance(2, stream=s.cuda_stream)  # resolves the kernel before the capture
    s.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        a.advance(2, stream=torch.cuda.current_stream().cuda_stream)
    for n in range(4):
        g.replay()
        torch.cuda.synchronize()
        if n % 2:
            a.advance(2)
            torch.cuda.synchronize()
    b.advance(2 + 4 * 2 + 2 * 2)
    for name in ("f", "g"):
        assert np.array_equal(a.valid(name), b.valid(name)), name
    a.close()
    b.close()
