"""Fields and several threads' copies around the sizes up to which a layout kernel
uses a pinned slot itself: 2^19 bytes with other calls beside it, a whole slot
alone.  The last field below, the first above, and one between the two.  Copies,
so bit for bit."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from opensayal_amd import Fluid
from tests.helpers import make_config

pytestmark = pytest.mark.gpu

SIZES = [(512, 256), (129, 1016), (513, 256), (500, 500)]


def there_and_back(W, H, seed):
    rng = np.random.default_rng(seed)
    with Fluid(make_config(W, H)) as fl:
        for _ in range(3):
            for name in ("vel_x", "smoke"):
                want = rng.integers(0, 0x7F800000, (H, W), dtype=np.uint32).view(np.float32)
                fl.set_field(name, want)
                if not np.array_equal(fl.get_field(name).view(np.uint32), want.view(np.uint32)):
                    return False
        return True


@pytest.mark.parametrize("W,H", SIZES)
def test_fields_at_the_limit(W, H):
    assert there_and_back(W, H, W)


def test_threads_at_the_limit():
    with ThreadPoolExecutor(6) as ex:
        assert all(ex.map(lambda i: there_and_back(*SIZES[i % 4], i), range(12)))
