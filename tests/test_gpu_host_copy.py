"""Fields read into memory of every kind a caller may pass."""
import time

import numpy as np
import pytest

import nimblesm_amd as N
from nimblesm_amd._capi import FIELDS, check, lib

pytestmark = pytest.mark.gpu


def model(num_nodes):
    """A model of one element and any number of nodes."""
    X = np.zeros((num_nodes, 3))
    X[:8] = [[0, 0, 0], [1, 0, 0], [1, 1, 0], [0, 1, 0], [0, 0, 1], [1, 0, 1], [1, 1, 1], [0, 1, 1]]
    m = N.ModelData(X, [N.Block(1, np.arange(8, dtype=np.int32)[None], N.NeohookeanMaterial(7800.0, 1.6e11, 0.8e11))])
    v = np.random.default_rng(num_nodes).normal(size=(num_nodes, 3))
    m.SetVectorNodeData("velocity", v)
    return m, v


def best(call, n=15):
    t = []
    for _ in range(n):
        t0 = time.perf_counter()
        call()
        t.append(time.perf_counter() - t0)
    return min(t)


@pytest.mark.parametrize("num_nodes", [100000, 625000, 2000000])
def test_pinned_and_device_destinations(hip_device, num_nodes):
    """A field of 2.4 to 48 MB into pinned memory, into the middle of it and
    into device memory: every value arrives, and pinned memory takes no longer
    than the runtime's own copy there (the bound, a quarter more, lies below
    the 1.4 to 2.3 times of a copy through further slots)."""
    import torch

    m, v = model(num_nodes)
    get = lambda p: check(lib().nsm_model_get_field(m._h, FIELDS["velocity"], p))  # noqa: E731
    pinned = torch.zeros(num_nodes * 3 + 7, dtype=torch.float64, pin_memory=True)
    for start in (0, 7):
        pinned.zero_()
        get(pinned.data_ptr() + 8 * start)
        assert np.array_equal(pinned.numpy()[start:start + 3 * num_nodes], v.ravel())
    dev = torch.zeros(num_nodes * 3, dtype=torch.float64, device=hip_device)
    torch.cuda.synchronize()
    get(dev.data_ptr())
    assert np.array_equal(dev.cpu().numpy(), v.ravel())
    here = pinned[:3 * num_nodes]

    def runtime():
        here.copy_(dev, non_blocking=True)
        torch.cuda.synchronize()

    assert best(lambda: get(pinned.data_ptr())) <= 1.25 * best(runtime)
    m.close()


@pytest.mark.parametrize("sizes", [(699050, 699051, 1398101), (1398102, 100000, 2500000)])
def test_copies_of_every_cut_in_turn(hip_device, sizes):
    """Fields on both sides of the sizes at which the cut changes (16 and 32
    MB), read by three threads at once, each in its own order: every value
    arrives, whichever pinned slots a copy finds."""
    import threading

    models = [model(n) for n in sizes]
    bad = []

    def read(k):
        for r in range(6):
            i = (k + r) % len(models)
            m, v = models[i]
            with locks[i]:  # one call of a model at a time
                got = m.GetVectorNodeData("velocity")
            if not np.array_equal(got, v):
                bad.append((k, i))

    locks = [threading.Lock() for _ in models]
    threads = [threading.Thread(target=read, args=(k,)) for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    for m, _ in models:
        m.close()
