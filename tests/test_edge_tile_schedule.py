"""CPU emulation of the register kernels' tiles at the grid's edges: the
first and last tiles of a row or column keep no halo there and own cells up to
the grid's edge, so (W - 4k) / tw tiles, rounded up, cover a row of W cells.
Every cell must be owned once, and sweeping each region on its own must
give the oracle's projection bit for bit.  With the halo one sweep too small
it must not."""
import numpy as np
import pytest

from oracle.oracle import OracleFluid
from tests.helpers import make_config, noise
from tests.test_resident_schedule import sweep_region
from tests.test_tiled_schedule import device_flags

f32 = np.float32


def spans(n, pitch, k, region):
    """(start, first owned, one past the last owned) of each tile of a row."""
    count = 1 if n <= 4 * k + pitch else -(-(n - 4 * k) // pitch)
    out = []
    for t in range(count):
        s = t * pitch
        out.append((s, s + (2 * k if t > 0 else 0),
                    s + 2 * k + pitch if t + 1 < count else n))
        assert n - s <= region or t + 1 < count
    return out


@pytest.mark.parametrize("region", [32, 64, 96, 128])
@pytest.mark.parametrize("k", [1, 2, 3, 5, 7])
def test_every_cell_is_owned_once(region, k):
    for n in range(1, 4 * region + 3):
        sp = spans(n, region - 4 * k, k, region)
        assert sp[0][1] == 0 and sp[-1][2] == n
        for (s, a, b), nxt in zip(sp, sp[1:] + [None]):
            assert a < b and a >= s and b <= s + region
            assert nxt is None or nxt[1] == b


def emulate(cfg, flags, u, v, k, rows, sweeps):
    H, W = u.shape
    for done in range(0, cfg.projection_n, sweeps):
        m = min(sweeps, cfg.projection_n - done)
        nu, nv = np.full_like(u, np.nan), np.full_like(v, np.nan)
        for gy, r0, r1 in spans(H, rows - 4 * k, k, rows):
            for gx, c0, c1 in spans(W, 128 - 4 * k, k, 128):
                jj, ii = np.mgrid[gy:gy + rows + 1, gx:gx + 129]
                inside = (ii < W) & (jj < H)
                jc, ic = np.minimum(jj, H - 1), np.minimum(ii, W - 1)
                F = np.where(inside, flags[jc, ic], 0).astype(np.int64)
                jc, ic, ins = jc[:rows, :128], ic[:rows, :128], inside[:rows, :128]
                U = np.where(ins, u[jc, ic], f32(0)).astype(f32)
                V = np.where(ins, v[jc, ic], f32(0)).astype(f32)
                sweep_region(cfg, F, U, V, None, gy, gx, m)
                nu[r0:r1, c0:c1] = U[r0 - gy:r1 - gy, c0 - gx:c1 - gx]
                nv[r0:r1, c0:c1] = V[r0 - gy:r1 - gy, c0 - gx:c1 - gx]
        u, v = nu, nv
    return u, v


@pytest.mark.parametrize("W,H,n,k,rows,drain", [(237, 77, 7, 5, 64, 1), (130, 70, 6, 3, 32, 0),
                                                (128, 64, 5, 2, 64, 1)])
def test_edge_tiles_match_oracle(W, H, n, k, rows, drain):
    cfg = make_config(W, H, projection_n=n, enable_drain=drain, obstacle_center_x=W // 2,
                      obstacle_center_y=H // 2, obstacle_radius=9.5)
    o = OracleFluid(cfg)
    o.set_state(u=noise((H, W), 51, 0.5), v=noise((H, W), 52, 0.5))
    flags, u, v = device_flags(o), o.u[::-1].copy(), o.v[::-1].copy()
    o.projection()

    def same(sweeps):
        gu, gv = emulate(cfg, flags, u, v, k, rows, sweeps)
        return (np.array_equal(gu[::-1].view(np.uint32), o.u.view(np.uint32)) and
                np.array_equal(gv[::-1].view(np.uint32), o.v.view(np.uint32)))

    assert same(k)
    if W > 128 or H > rows:  # a planted mistake: a sweep more than the halo is good for
        assert not same(k + 1)
