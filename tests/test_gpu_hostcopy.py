"""Host transfers of a context (fx_state_upload / fx_state_download): bytes unchanged at sizes around
the threshold of the staged copy and around its chunks, from read-only and from new arrays, and with
several contexts transferring at once from threads of their own."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from fluxo_amd.mesh import box_mesh
from fluxo_amd.native import Engine

pytestmark = pytest.mark.gpu

NODE_BYTES = 64 * 40  # an element at N = 3
MIB = 1 << 20


def context(elements):
    m = box_mesh((elements, 1, 1), 3, length=(float(elements), 1.0, 1.0))
    return Engine(m)


def random_state(e, seed):
    U = np.random.default_rng(seed).standard_normal(e.shape())
    U.setflags(write=False)
    return U


def busy_context():
    """A context whose transfers have had the device's copying threads made."""
    e = context(40 * MIB // NODE_BYTES)
    U = random_state(e, 5)
    e.upload(U)
    assert np.array_equal(e.download(), U)
    return e


@pytest.fixture
def workers():
    e = busy_context()
    yield
    e.close()


@pytest.mark.usefixtures("workers")
@pytest.mark.parametrize("nbytes", [64 << 10, 4 * MIB, 5 * MIB, 8 * MIB, 9 * MIB, 33 * MIB])
@pytest.mark.parametrize("step", [0, 1])
def test_state_round_trip(nbytes, step):
    e = context(nbytes // NODE_BYTES + step)  # the last size below and the first above
    for seed in (1, 2):
        U = random_state(e, seed)
        e.upload(U)
        assert np.array_equal(e.download(), U)
    e.close()


def test_contexts_transfer_at_once():
    first = busy_context()
    es = [context(7000 + 7 * i) for i in range(3)]

    def work(e, seed):
        same = 0
        for r in range(4):
            U = random_state(e, 10 * seed + r)
            e.upload(U)
            same += np.array_equal(e.download(), U)
        return same

    with ThreadPoolExecutor(len(es)) as pool:  # result() raises what a transfer raised
        assert [f.result() for f in [pool.submit(work, e, i) for i, e in enumerate(es)]] == [4, 4, 4]
    for e in [first] + es:
        e.close()
    busy_context().close()  # the workers are made again after the last context gave them back
