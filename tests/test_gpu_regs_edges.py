"""The register-resident projection kernels where their tiles meet the grid:
wavefronts of every kind (all open, a wall down the rows, an odd or an even
drain column, anything else), tiles that own cells up to the grid's edge, one
tile and one cell more than one tile, launches of every region height, and
the pressure quotient by reciprocal and by division.  Bit for bit against the
oracle (a copy of the reference's update rule, so there is no tolerance)."""
import numpy as np
import pytest

from opensayal_amd import Batch, Fluid
from tests.helpers import make_config
from tests.test_gpu_parity import assert_bitwise, pair

pytestmark = pytest.mark.gpu


def shape(kernel, rows, k):
    return dict(projection_kernel=kernel, tile_width=128 - 4 * k, tile_height=8 * rows - 4 * k,
                sweeps_per_launch=k)


# grid, options: what the right and top tiles hold
GRIDS = [
    (128, 96, {}),                                # one tile of 96 rows, odd drain column
    (129, 97, {}),                                # one cell over it, even drain column
    (237, 165, {}),                               # 128 + 108 + 1 columns at k = 5
    (236, 165, dict(enable_drain=0)),             # a closed wall in an odd column
    (345, 141, dict(enable_drain=0)),             # and in an even one
    (200, 133, dict(obstacle_center_x=110, obstacle_center_y=64, obstacle_radius=31.0)),
]


@pytest.mark.parametrize("W,H,opts", GRIDS)
@pytest.mark.parametrize("kernel,rows,k", [(2, 4, 3), (2, 8, 5), (2, 10, 4), (2, 12, 5),
                                           (2, 16, 6), (3, 4, 3), (3, 8, 4), (3, 12, 5)])
def test_edge_tiles(W, H, opts, kernel, rows, k):
    cfg = make_config(W, H, wind_speed=2.0, g=-5.0, projection_n=11, **opts)
    fl, o = pair(cfg, seed=31)
    fl.set_tuning(**shape(kernel, rows, k))
    fl.step(2)
    o.update(steps=2)
    assert_bitwise(fl, o, f"{W}x{H} kernel {kernel} rows {rows} k {k}")


@pytest.mark.parametrize("d_t,density,cell_size", [(0.05, 1.0, 1.0), (0.05, 1.3, 2.0),
                                                   (2.5, 1.0, 1.0)])
@pytest.mark.parametrize("kernel,rows", [(2, 4), (2, 8), (3, 4), (3, 8)])
def test_edge_tiles_pressure(d_t, density, cell_size, kernel, rows):
    """Unit, reciprocal and dividing pressure quotients, from a field that
    is not 0 (the projection alone adds to it) and over whole steps."""
    cfg = make_config(237, 133, projection_n=7, enable_pressure=1, wind_speed=0.5, d_t=d_t,
                      density=density, cell_size=cell_size)
    fl, o = pair(cfg, seed=32)
    fl.set_tuning(**shape(kernel, rows, 4))
    p = np.random.default_rng(5).uniform(-1, 1, (133, 237)).astype(np.float32)
    fl.set_field("pressure", p)
    o.set_state(p=p)
    fl.project()
    o.projection()
    assert_bitwise(fl, o, "projection")
    fl.step(2)
    o.update(steps=2)
    assert_bitwise(fl, o, "steps")


@pytest.mark.parametrize("storage", [1, 2])  # binary16, bfloat16
@pytest.mark.parametrize("kernel,rows", [(2, 8), (2, 12), (3, 4), (3, 12)])
def test_edge_tiles_16_bit(storage, kernel, rows):
    """Every shape rounds as the colour-phase kernel does."""
    out = []
    for tuning in (dict(projection_kernel=0), shape(kernel, rows, 4)):
        cfg = make_config(237, 133, projection_n=9, wind_speed=2.0, storage=storage)
        fl, _ = pair(cfg, seed=33)
        fl.set_tuning(**tuning)
        fl.step(2)
        out.append([fl.get_field(n).view(np.uint32) for n in ("vel_x", "vel_y", "smoke")])
    for a, b in zip(*out):
        assert np.array_equal(a, b)


def test_batch_member_with_a_dividing_pressure():
    """A member whose pressure needs the division steps beside the others."""
    cfgs = [make_config(150, 100, projection_n=9, enable_pressure=1, wind_speed=0.5, d_t=d_t)
            for d_t in (2.5, 0.05)]
    made = [pair(c, seed=34 + i) for i, c in enumerate(cfgs)]
    with Batch() as bt:
        for fl, _ in made:
            bt.add(fl)
        bt.step(3)
        for fl, o in made:
            o.update(steps=3)
            assert_bitwise(fl, o, f"d_t {o.cfg.d_t}")
