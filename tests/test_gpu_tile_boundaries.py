"""The tile step's second loads: sources that are not read directly (walls,
slip walls, solid cells, wall ghosts behind an OUTFLOW face) are loaded again
lane by lane, PRESSURE and inlet ghosts take their constants.  Against the
row-block kernels, whose pull resolves every source before its loads: the same
arithmetic on the same values, so the results are equal bit for bit.  The
large shapes (2^18 cells and more) take the FP64 step in one launch, in each
of its boundary instances: no table or pressure, a profile inlet at y-lo,
PRESSURE faces, and both."""
import numpy as np
import pytest

from marbles_amd import configs

pytestmark = pytest.mark.gpu

BLOCKS = "k_qpass+k_collide"
TILES = "k_qpass_x256+k_collide_x256"  # FP64 arithmetic in every storage


def _walled(n, lo, hi):
    """A sphere in a box with the given faces (1 wall, 5 outflow, 6/7/8 slip
    normal to x/y/z), the flow started at Mach 0.05 along x."""
    cfg = configs.channel_sphere(n, radius=3.5, center=(6.0, 6.0, 6.0), tau=0.7)
    cfg.update(periodic=(0, 0, 0), bc_lo=lo, bc_hi=hi)
    return cfg


CASES = {
    "walls": lambda n: _walled(n, (1, 1, 1), (1, 1, 1)),
    # wall ghosts behind y and z OUTFLOW faces, a velocity inlet beside them
    "open_corners": lambda n: _walled(n, (2, 1, 5), (5, 5, 1)),
    "open_z": lambda n: _walled(n, (1, 5, 5), (6, 1, 5)),
    "slip": lambda n: configs.slip_channel(n),
    "duct": lambda n: configs.channel_profile(n),
    "y_inlet": lambda n: dict(configs.channel_profile(n), bc_lo=(1, 2, 1), bc_hi=(1, 5, 1)),
    "pressure_outlet": lambda n: configs.pressure_case("outlet", n),
    "pressure_both": lambda n: configs.pressure_case("both", n),
    "pressure_channel": lambda n: configs.pressure_case("channel", n),
}


@pytest.mark.parametrize("storage,shape", [("f64", (37, 19, 14)), ("f32s", (37, 19, 14)), ("f16s", (37, 19, 14)),
                                           ("f64", (131, 47, 45))])
@pytest.mark.parametrize("case", sorted(CASES))
def test_tile_step_equals_row_blocks_at_boundaries(engine, case, storage, shape):
    out = []
    for variant in (TILES, BLOCKS):
        E = configs.build_level(CASES[case](shape), layout="compact", storage=storage)
        E.set_hot_kernel(variant)
        E.advance(5)
        out.append([E.valid(name) for name in ("f", "g")])
        E.close()
    for a, b in zip(*out):
        assert np.isfinite(a).all() and np.array_equal(a, b), (case, storage, shape)


@pytest.mark.parametrize("case", ["walls", "open_corners", "duct", "y_inlet"])
def test_fp32_arithmetic_tile_step_equals_row_blocks_at_boundaries(engine, case):
    """The shifted FP32 storage's default step (FP32 arithmetic in pass 2)."""
    out = []
    for variant in ("k_qpass_x256+k_collide_f32_x256", "k_qpass_y2+k_collide_f32"):
        E = configs.build_level(CASES[case]((37, 19, 14)), layout="compact", storage="f32s")
        E.set_hot_kernel(variant)
        E.advance(5)
        out.append([E.valid(name) for name in ("f", "g")])
        E.close()
    for a, b in zip(*out):
        assert np.isfinite(a).all() and np.array_equal(a, b), case


@pytest.mark.parametrize("case", ["walls", "open_corners", "duct", "y_inlet"])
def test_fp16_default_step_equals_row_blocks_at_boundaries(engine, case):
    """The scaled FP16 storage's default step (FP32 arithmetic in pass 2 on
    tiles): the row-block variant launches its own kernel, with the same scales
    and box maxima."""
    out = []
    for variant in (None, "k_qpass_x256+k_collide_h32_x256"):
        E = configs.build_level(CASES[case]((37, 19, 14)), layout="compact", storage="f16s")
        if variant:
            E.set_hot_kernel(variant)
        E.advance(12)
        out.append([E.valid(name) for name in ("f", "g")])
        E.close()
    for a, b in zip(*out):
        assert np.isfinite(a).all() and np.array_equal(a, b), case


def test_full_size_y_inlet_deck_equals_row_blocks(engine):
    """The 246 x 576 x 4 cylinder deck with its parabolic inlet at y-lo."""
    out = []
    for variant in (TILES, BLOCKS):
        E = configs.build_level(configs.cylinder_deck("single_cylinder"), layout="compact")
        E.set_hot_kernel(variant)
        E.advance(5)
        out.append([E.valid(name) for name in ("f", "g")])
        E.close()
    for a, b in zip(*out):
        assert np.isfinite(a).all() and np.array_equal(a, b)


@pytest.mark.parametrize("storage,shape,variant,launches", [
    ("f64", (37, 19, 14), None, "k_qpass_tile+k_collide_tile"),
    ("f64", (131, 47, 45), None, "k_step"),
    ("f64", (131, 47, 45), "k_qpass_x128+k_collide_x128", "k_qpass_x128+k_collide_x128"),
    ("f32s", (131, 47, 45), None, "k_qpass_tile+k_collide_tile"),
    ("f16s", (131, 47, 45), None, "k_qpass_tile+k_collide_tile_w4"),
    ("f16s", (37, 19, 14), "k_qpass_x256+k_collide_h32_x256", "k_qpass_x256+k_collide_h32_x256"),
])
def test_timed_steps_name_the_kernels_that_run(engine, storage, shape, variant, launches):
    """One slot per launched kernel, under its own name, each with a time."""
    E = configs.build_level(CASES["walls"](shape), layout="compact", storage=storage)
    if variant:
        E.set_hot_kernel(variant)
    assert E.hot_kernel_launches() == launches
    ms = E.advance_timed(3)
    assert list(ms) == launches.split("+") and all(t > 0.0 for t in ms.values()), ms
    E.close()


@pytest.mark.parametrize("variant", [TILES, "k_sweep", "k_sweep_x64"])
def test_steps_that_wait_between_blocks_report_no_fault(engine, variant):
    """k_step and the z-sweeps count the bounded waits that ran out; the count
    starts at zero and a step that went well leaves it there."""
    E = configs.build_level(CASES["walls"]((131, 47, 45)), layout="compact")
    assert E.step_faults() == 0
    E.set_hot_kernel(variant)
    E.advance(4)
    assert E.step_faults() == 0 and np.isfinite(E.valid("f")).all()
    E.close()
