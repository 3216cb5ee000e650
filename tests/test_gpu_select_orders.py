"""Selection among values in a regular order: the sample that brackets the rank
must not alias with the order, so such calls take the path that randomly
ordered values take (and its time)."""
import ctypes as C

import numpy as np
import pytest
import torch

from multilanguagekdtree_amd import _lib

pytestmark = pytest.mark.gpu


def select(vals, goal):
    """Indices partitioned around the goal, and the best of ten times in ms."""
    n = len(vals)
    L = _lib.lib()
    dv = torch.as_tensor(vals, device="cuda")
    base = torch.arange(n, dtype=torch.int64, device="cuda")
    ix = torch.empty_like(base)
    size = int(L.kd_quickstat_workspace_bytes(n))
    ws = torch.empty(size, dtype=torch.uint8, device="cuda")
    best = float("inf")
    a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    for _ in range(10):
        ix.copy_(base)
        torch.cuda.synchronize()
        a.record()
        _lib.check(L.kd_quickstat_index_device(n, C.c_void_p(ix.data_ptr()), goal,
                                               C.c_void_p(dv.data_ptr()), n,
                                               C.c_void_p(ws.data_ptr()), size))
        b.record()
        torch.cuda.synchronize()
        best = min(best, a.elapsed_time(b))
    return ix.cpu().numpy(), best


def expected(vals, goal):
    order = np.lexsort((np.arange(len(vals)), vals))
    rank = np.empty(len(vals), np.int64)
    rank[order] = np.arange(len(vals))
    every = np.arange(len(vals))
    return np.concatenate([every[rank < goal], [order[goal]], every[rank > goal]])


def ordered_values(kind, n):
    i = np.arange(n)
    return {"fastest": lambda: i % 128 + 0.0,          # a lattice's fastest coordinate
            "saw": lambda: i % 256 + i / n,            # the same, distinct values
            "middle": lambda: i // 128 % 128 + 0.0,
            "alternating": lambda: (i & 1) + 0.0,
            "sorted": lambda: i + 0.0,
            "reversed": lambda: n - i - 0.0}[kind]()


@pytest.mark.parametrize("kind", ["fastest", "saw", "middle", "alternating", "sorted", "reversed"])
@pytest.mark.parametrize("n", [8192, 8193, 1 << 17, 128 ** 3])
def test_partition(kind, n):
    vals = ordered_values(kind, n)
    for goal in (0, n // 3, n // 2, n - 1):
        np.testing.assert_array_equal(select(vals, goal)[0], expected(vals, goal))


@pytest.mark.parametrize("kind", ["fastest", "saw", "alternating"])
def test_time_does_not_depend_on_the_order(kind):
    # (a bracket that misses costs the radix passes on top: 2.5 times as much)
    n = 1 << 22
    vals = ordered_values(kind, n)
    shuffled = np.random.default_rng(1).permutation(vals)
    goal = int(0.37 * n)
    t, ref = select(vals, goal)[1], select(shuffled, goal)[1]
    assert t <= 1.6 * ref
