"""The pinned arrays that logits are returned in: never shared by two results that are alive, reused once released, bounded, freed when closed
(the allocator is the C heap here: no GPU)."""
import ctypes as C
import gc
import threading

import numpy as np

from vllm_rs_amd.engine import _PinnedPool


class Heap:
    def __init__(self, fail=False):
        self.blocks, self.fail = {}, fail

    def vra_malloc_host(self, n):
        if self.fail:
            return None
        b = C.create_string_buffer(n)
        self.blocks[C.addressof(b)] = b
        return C.addressof(b)

    def vra_free_host(self, p):
        del self.blocks[p]

    def vra_clear_error(self):
        pass


def test_results_that_are_alive_share_nothing():
    heap = Heap()
    pool = _PinnedPool(heap)
    kept = []
    for i in range(20):
        a = pool.take((3, 1000))
        a[:] = i
        kept.append(a[1:] if i % 2 else a)  # (a view keeps the memory, too)
        del a
    assert all((a == i).all() for i, a in enumerate(kept)) and len(heap.blocks) == 20
    del kept
    gc.collect()
    again = [pool.take((3, 1000)) for _ in range(20)]
    assert len(heap.blocks) == 20 and len({a.ctypes.data for a in again}) == 20 and all(a.dtype == np.float32 and a.flags.writeable for a in again)


def test_bounds_and_close():
    heap = Heap()
    pool = _PinnedPool(heap)
    pool.LIVE, pool.KEEP = 1 << 20, 1 << 18
    arrays = [pool.take((1 << 15,)) for _ in range(12)]  # 128 KiB each: eight are pinned
    assert len(heap.blocks) == 8 and pool.live == 1 << 20
    assert pool.take((0, 5)).shape == (0, 5) and pool.take((1 << 20,)).size == 1 << 20 and len(heap.blocks) == 8
    one = arrays[0]
    del arrays
    gc.collect()
    assert len(heap.blocks) == 3 and pool.idle == 1 << 18  # two idle and the one in use
    pool.close()
    assert len(heap.blocks) == 1 and pool.take((4,)).size == 4 and len(heap.blocks) == 1
    one[:] = 1.0
    del one
    gc.collect()
    assert not heap.blocks and pool.live == 0
    assert _PinnedPool(Heap(fail=True)).take((2, 2)).shape == (2, 2)


def test_threads():
    heap = Heap()
    pool = _PinnedPool(heap)
    bad = []

    def work(seed):
        for i in range(300):
            a = pool.take((64 + seed, 17))  # (beside the last one: two a thread)
            a[:] = seed
            if not (a == seed).all():
                bad.append(seed)

    threads = [threading.Thread(target=work, args=(s,)) for s in range(6)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    gc.collect()
    assert not bad and len(heap.blocks) <= 12 and pool.live == sum(len(b) for b in heap.blocks.values())
