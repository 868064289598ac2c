"""CPU emulation of the row exchange between a tile's wavefronts as the register,
resident and batch projection kernels have it (reg_phase in
projection_device.hpp): one barrier per colour phase.  Each wavefront publishes
its row 0 after computing, without the update from below, beside the update that
its last row makes to the row above, and applies the one from below in the next
phase.  The row it reads lacks that update too, but only in the cells that its own
last row does not touch in that phase.  Wavefronts sit out the phases in which
none of their rows reaches the tile.  The owned rows must equal, bit for bit, those
of sweeping the region as a whole; with a row read a phase late they must not."""
import numpy as np
import pytest

from oracle.oracle import OracleFluid
from tests.helpers import make_config, noise
from tests.test_resident_schedule import CF_FU, CF_FV, CF_UPD, sweep_region
from tests.test_tiled_schedule import device_flags

f32 = np.float32


class Wave:
    def __init__(self, cfg, F, U, V, w, R, NW):
        self.w, self.R, self.NW, self.o = w, R, NW, f32(cfg.projection_o)
        rows = slice(w * R, w * R + R)
        self.F, self.u, self.v = F[w * R:w * R + R + 1], U[rows].copy(), V[rows].copy()

    def row(self, r, colour, above):
        """apply_projection_at for the active cells of row r; `above` is row 0 of
        the wavefront above.  Returns the update of the row above."""
        width = self.u.shape[1]
        q = np.arange(colour, width, 2)
        f = self.F[r, q].astype(np.int64)
        upd = (f & CF_UPD) != 0
        top = self.v[r + 1] if r + 1 < self.R else above
        right = np.append(self.u[r], f32(0))
        uu, vv, ur, vt = self.u[r, q], self.v[r, q], right[q + 1], top[q]
        div = (((ur - uu).astype(f32) + vt).astype(f32) - vv).astype(f32)
        with np.errstate(divide="ignore", invalid="ignore"):
            d = (self.o * (div / ((f >> 4) & 7).astype(f32)).astype(f32)).astype(f32)
        d = np.where(upd, d, f32(0))

        def gated(flag):
            return np.where(upd & flag, d, f32(0))

        dl, dr = gated((f & CF_FU) != 0), gated((self.F[r, q + 1] & CF_FU) != 0)
        db, dt = gated((f & CF_FV) != 0), gated((self.F[r + 1, q] & CF_FV) != 0)
        inside = q + 1 < width
        self.u[r, q] = (uu + dl).astype(f32)
        self.u[r, q[inside] + 1] = (ur - dr).astype(f32)[inside]
        self.v[r, q] = (vv + db).astype(f32)
        if r + 1 < self.R:
            self.v[r + 1, q] = (vt - dt).astype(f32)
            return None
        send = np.zeros(width, f32)
        send[q] = dt
        return send

    def settle(self):
        self.v[0] = (self.v[0] - self.from_below).astype(f32)

    def phase(self, colour, active):
        """colour: parity of the active columns of row 0."""
        self.sent = np.zeros(self.u.shape[1], f32)
        if not active:
            self.settle()
            return
        for r in range(1, self.R - 1):
            self.row(r, (colour + r) & 1, None)
        self.settle()
        self.row(0, colour, None)
        self.sent = self.row(self.R - 1, (colour + self.R - 1) & 1, self.read)


def sweep_waves(cfg, F, U, V, R, NW, gy0, sweeps, r0, r1, late=False):
    waves = [Wave(cfg, F, U, V, w, R, NW) for w in range(NW)]
    none = np.zeros(U.shape[1], f32)
    held = []

    def exchange():  # the barrier lies between what is written and what is read
        rows, sent = [x.v[0].copy() for x in waves], [x.sent for x in waves]
        if late:
            rows, held[:] = list(held) or rows, rows
        for w, x in enumerate(waves):
            x.from_below = sent[w - 1] if w > 0 else none
            x.read = rows[w + 1] if w + 1 < NW else none

    for x in waves:
        x.sent = none
    exchange()
    for ph in range(2 * sweeps):
        for x in waves:
            base = x.w * R
            idle = max(r0 - base - R, base - r1 + 1, 0)
            active = ph < 2 * (max(2 * sweeps - idle + 1, 0) // 2)
            x.phase((ph + gy0 + base) & 1, active)
        exchange()
    for x in waves:
        x.settle()
    return np.concatenate([x.u for x in waves]), np.concatenate([x.v for x in waves])


@pytest.mark.parametrize("R,NW,k", [(4, 8, 2), (8, 8, 5), (10, 8, 3), (6, 16, 7), (8, 16, 1)])
@pytest.mark.parametrize("gx,gy", [(0, 0), (40, 36)])
def test_exchange_equals_the_whole_region(R, NW, k, gx, gy):
    H, W = NW * R + 60, 200
    cfg = make_config(W, H, projection_n=k, obstacle_center_x=gx + 60,
                      obstacle_center_y=gy + NW * R // 2, obstacle_radius=9.5)
    o = OracleFluid(cfg)
    flags = device_flags(o)
    rows, cols = NW * R, 128
    F = flags[gy:gy + rows + 1, gx:gx + cols + 1].astype(np.int64)
    U = noise((H, W), 71, 0.5).astype(f32)[gy:gy + rows, gx:gx + cols].copy()
    V = noise((H, W), 72, 0.5).astype(f32)[gy:gy + rows, gx:gx + cols].copy()
    r0, r1 = (2 * k if gy else 0), rows - 2 * k
    want_u, want_v = U.copy(), V.copy()
    sweep_region(cfg, F, want_u, want_v, None, gy, gx, k)

    def same(late):
        u, v = sweep_waves(cfg, F, U, V, R, NW, gy, k, r0, r1, late)
        return (np.array_equal(u[r0:r1].view(np.uint32), want_u[r0:r1].view(np.uint32)) and
                np.array_equal(v[r0:r1].view(np.uint32), want_v[r0:r1].view(np.uint32)))

    assert same(False)
    assert not same(True)  # a planted mistake
