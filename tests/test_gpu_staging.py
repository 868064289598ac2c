"""Fields in and out through pinned slots of 1 MB: one slot exactly, one cell
more, every slot, more chunks than slots; pageable, pinned and unaligned
host memory; calls from several threads at once.  Copies, so bit for bit."""
import ctypes
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from opensayal_amd import Fluid, _abi
from tests.helpers import make_config

pytestmark = pytest.mark.gpu


def bits(rng, W, H):
    return rng.integers(0, 0x7F800000, (H, W), dtype=np.uint32).view(np.float32)


def there_and_back(W, H, seed):
    rng = np.random.default_rng(seed)
    with Fluid(make_config(W, H)) as fl:
        want = {n: bits(rng, W, H) for n in ("vel_x", "vel_y", "smoke")}
        for n, a in want.items():
            fl.set_field(n, a)
        return all(np.array_equal(fl.get_field(n).view(np.uint32), a.view(np.uint32))
                   for n, a in want.items())


@pytest.mark.parametrize("W,H", [(3, 3), (512, 512), (513, 512), (1021, 771), (1024, 1024),
                                 (1025, 1025), (2051, 1537)])
def test_fields_survive_the_slots(W, H):
    assert there_and_back(W, H, W)


def test_threads_do_not_share_a_slot():
    sizes = [(64, 36), (512, 512), (1025, 1025), (700, 300)] * 3
    with ThreadPoolExecutor(6) as ex:
        assert all(ex.map(lambda i: there_and_back(*sizes[i], i), range(len(sizes))))


@pytest.mark.parametrize("W,H", [(64, 36), (1025, 513)])
def test_pinned_and_unaligned_host_memory(W, H):
    want = bits(np.random.default_rng(7), W, H)
    with Fluid(make_config(W, H)) as fl:
        fl.set_field("vel_x", want)
        fid = 0  # OSY_FIELD_VEL_X
        hip = ctypes.CDLL("libamdhip64.so.7")  # the runtime already loaded
        pinned = ctypes.c_void_p()
        assert hip.hipHostMalloc(ctypes.byref(pinned), ctypes.c_size_t(want.nbytes), 0) == 0
        raw = np.zeros(want.nbytes + 1, np.uint8)
        for at in (pinned.value, raw.ctypes.data + 1):
            _abi.check(_abi.lib().osy_fluid_get_field(fl._h, fid, ctypes.c_void_p(at),
                                                      want.nbytes))
        assert ctypes.string_at(pinned.value, want.nbytes) == want.tobytes()
        assert raw[1:].tobytes() == want.tobytes()
        assert hip.hipHostFree(pinned) == 0
