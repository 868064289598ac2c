"""A resident projection that the caller captures into a graph: replayed several
times, with the handle's own projections in the same and in another resident
shape between, it gives the bits of projections alone."""
import ctypes

import numpy as np
import pytest

from opensayal_amd import Fluid, Stream, workloads as wl
from tests.helpers import make_config

pytestmark = pytest.mark.gpu


def fields(fl):
    return [fl.get_field(n).view(np.uint32) for n in ("vel_x", "vel_y", "pressure")]


@pytest.mark.parametrize("pressure", [0, 1])
def test_captured_resident_projection_replays(pressure):
    hip = ctypes.CDLL("libamdhip64.so.7")  # the runtime already loaded
    cfg = make_config(250, 230, projection_n=13, enable_pressure=pressure,
                      obstacle_center_x=100, obstacle_center_y=104, obstacle_radius=20.5)
    u, v, _ = wl.initial_state(cfg, 5)
    shapes = [dict(projection_kernel=3, tile_width=108, tile_height=44, sweeps_per_launch=5),
              dict(projection_kernel=3, tile_width=120, tile_height=24, sweeps_per_launch=2)]
    with Fluid(cfg) as fl, Fluid(cfg) as plain:
        stream = Stream()
        for f in (fl, plain):
            f.set_field("vel_x", u)
            f.set_field("vel_y", v)
        fl.set_tuning(**shapes[0])
        handle = ctypes.c_void_p(stream.handle)
        graph, run = ctypes.c_void_p(), ctypes.c_void_p()
        assert hip.hipStreamBeginCapture(handle, 1) == 0  # hipStreamCaptureModeThreadLocal
        fl.project(stream=stream, sync=False)
        assert hip.hipStreamEndCapture(handle, ctypes.byref(graph)) == 0
        assert hip.hipGraphInstantiate(ctypes.byref(run), graph, None, None,
                                       ctypes.c_size_t(0)) == 0

        def replay():
            assert hip.hipGraphLaunch(run, handle) == 0
            stream.synchronize()

        # a launch reads the buffers the state lay in at the capture and writes
        # the others, where it lies for the handle since
        plain.project()
        replay()
        for got, want in zip(fields(fl)[:2], fields(plain)):
            assert np.array_equal(got, want)
        for shape in (shapes[0], shapes[1], shapes[0]):
            fl.set_tuning(**shape)
            for _ in range(2):  # back to the buffers the graph reads, and on
                fl.project()
                plain.project()
            want = fields(plain)
            for got, ref in zip(fields(fl), want):
                assert np.array_equal(got, ref)
            replay()  # the last of those once more: the same but for its sums
            for got, ref in zip(fields(fl)[:2], want):
                assert np.array_equal(got, ref)
            for f in (fl, plain):  # the sums of both from here
                f.set_field("pressure", np.zeros((230, 250), np.float32))
        assert hip.hipGraphExecDestroy(run) == 0 and hip.hipGraphDestroy(graph) == 0
        stream.close()
