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


def counted(pool):
    pool.L.taken = 0
    real = pool.L.vra_malloc_host

    def take(n):
        pool.L.taken += 1
        return real(n)

    pool.L.vra_malloc_host = take
    return pool


def test_repeated_large_results_are_pinned_once():
    """a loop that holds the last result while the next one is made (two alive), and one that releases it first: results of more than KEEP are no more
    pinned anew at every call than small ones, and no more than an eighth beyond their size is pinned for them"""
    for rows in (3, 80, 262):
        pool = counted(_PinnedPool(Heap()))
        pool.LIVE, pool.KEEP = 1 << 25, 1 << 20
        nbytes = rows * 8016 * 4
        for _ in range(6):
            pool.take((rows, 8016))
        assert pool.L.taken == 1, rows
        out = None
        for _ in range(6):
            out = pool.take((rows, 8016))
        assert pool.L.taken <= 2 and all(len(b) <= max(nbytes * 9 // 8, 2 * nbytes if nbytes < 1 << 20 else 0, 1 << 17) for b in pool.L.blocks.values())
        del out
        assert pool.idle <= max(pool.KEEP, nbytes * 9 // 8) and len(pool.L.blocks) in (1, 2)


def test_idle_memory_makes_room():
    """memory that is idle does not stand in the way of a result that needs other memory, and a buffer that was given back is the last to go"""
    pool = counted(_PinnedPool(Heap()))
    pool.LIVE, pool.KEEP = 1 << 23, 1 << 22
    small = [pool.take((1 << 18,)) for _ in range(6)]  # 1 MiB each
    del small
    gc.collect()
    assert pool.idle == 1 << 22 and pool.live == 1 << 22
    big = pool.take((7 << 18,))  # 7 MiB: three of the four idle ones go
    assert pool.live == 1 << 23 and pool.idle == 1 << 20 and len(pool.L.blocks) == 2
    del big
    assert pool.idle == 7 << 20 and len(pool.L.blocks) == 1
    pool.close()
    assert not pool.L.blocks and pool.live == 0
