"""GPU tests of the copy kernels at the edges of their tiles.

A kernel-mode save into, or load out of, a buffer in device memory moves each
chunk as units of one wave; one that crosses the host link takes tiles from a
queue.  The sizes here sit at the edges of a unit or a tile
(one wave's words, one more, one less), of a workgroup's share, of the
descriptor table that small calls read in place, and of a launch.  The expected
bytes are a numpy indexing of the same layout.
"""

import threading

import numpy as np
import pytest

from pegaflow_amd import _lib
from pegaflow_amd.runtime import DeviceBuffer, PinnedBuffer, host_wait_word
from pegaflow_amd.transfer import (KVCacheRegistration, LayerTransfer, TransferContext,
                                   block_array)

pytestmark = pytest.mark.gpu


class Layer:
    """A KV tensor of ``nb`` blocks in ``segs`` segments of ``bpb`` bytes, and the
    ``ids`` that move between it and a buffer holding a K and a V region."""

    def __init__(self, nb, bpb, segs, ids, seed):
        self.shape, self.ids = (segs, nb, bpb), np.asarray(ids, np.int64)
        self.dev = DeviceBuffer((segs * nb * bpb + 7) // 8 * 8)
        self.dev.fill_random(seed)
        self.host = self.dev.download()
        self.reg = KVCacheRegistration.create(self.dev.ptr, segs * nb * bpb, nb, bpb,
                                              nb * bpb if segs == 2 else 0, segs)
        self.nbytes = segs * len(self.ids) * bpb

    def view(self, flat):
        segs, nb, bpb = self.shape
        return flat[:segs * nb * bpb].reshape(self.shape)

    def transfer(self, base):
        segs, _, bpb = self.shape
        at = base + np.arange(len(self.ids), dtype=np.uint64) * np.uint64(bpb)
        v = at + np.uint64(len(self.ids) * bpb) if segs == 2 else None
        return LayerTransfer(self.reg, block_array(self.ids, at, v))

    def packed(self):
        return self.view(self.host)[:, self.ids].reshape(-1)

    def restore(self, packed):
        segs, _, bpb = self.shape
        self.view(self.host)[:, self.ids] = packed.reshape(segs, len(self.ids), bpb)


def make_layers(rng, bpb, segs, counts, nb):
    return [Layer(nb, bpb, segs, rng.choice(nb, n, replace=False), 10 + i)
            for i, n in enumerate(counts)]


def bases(layers, base):
    out = []
    for l in layers:
        out.append(base)
        base += l.nbytes
    return out


# Segment sizes around a wave's words (1 KiB) and its unit (2 KiB), and one of
# many units; layers of none, one and several blocks.
MARKED = [(bpb, 2, (3, 0, 1, 17), 40, cap)
          for bpb in (16, 1008, 1024, 1040, 2032, 2048, 2064, 8208, 36864) for cap in (0, 3)]
# Launches large enough for the larger shares of a workgroup, blocks-first and split.
MARKED += [(32768, 2, (300, 301), 400, 0), (36864, 1, (511, 1, 512), 600, 0)]
# A launch with a workgroup's middle share (layers of 2 MiB and more, or 32 MiB in all).
MARKED += [(4096, 1, (700,), 800, 0), (36864, 1, (100, 99) * 5, 120, 7)]
# More layers than a workgroup has lanes.
MARKED += [(1040, 2, (1, 0, 3) * 180, 20, 0), (1040, 2, (1, 0, 3) * 180, 20, 5)]


@pytest.mark.parametrize("bpb,segs,counts,nb,cap", MARKED)
def test_marked_load_from_device_memory(gpu, bpb, segs, counts, nb, cap):
    """One marked launch over the layers: every byte and every word, twice (the
    layers' counters are 0 again after a launch)."""
    rng = np.random.default_rng(bpb + cap)
    layers = make_layers(rng, bpb, segs, counts, nb)
    pool = DeviceBuffer(sum(l.nbytes for l in layers))
    words, dev_words = PinnedBuffer(8 * len(layers)), DeviceBuffer(8 * len(layers))
    words.array[:] = 0
    dev_words.memset(0)
    ctx = TransferContext(0)
    ctx.set_max_grid(cap)
    for value in (1, 2):
        pool.fill_random(100 + value, nbytes=pool.nbytes // 8 * 8)
        packed = pool.download()
        ctx.load_layers_marked([l.transfer(b) for l, b in zip(layers, bases(layers, pool.ptr))],
                               [(words.ptr, value, True), (dev_words.ptr, value, False)],
                               _lib.MODE_KERNEL)
        ctx.synchronize()
        assert words.array.view(np.uint64).tolist() == [value] * len(layers)
        assert dev_words.download().view(np.uint64).tolist() == [value] * len(layers)
        for l, at in zip(layers, bases(layers, 0)):
            l.restore(packed[at:at + l.nbytes])
            assert np.array_equal(l.dev.download(), l.host)
    ctx.close()


@pytest.mark.parametrize("bpb", [65536, 65537])
def test_large_marked_layers_have_a_launch_each(gpu, bpb):
    """Layers of 96 MiB and more among smaller and empty ones: every byte, every word, and
    the copies that it took."""
    counts = (2, 800, 0, 1, 767, 768)  # 96 MiB are 768 blocks of 2 x 64 KiB
    layers = make_layers(np.random.default_rng(bpb), bpb, 2, counts, 804)
    pool, words = DeviceBuffer(sum(l.nbytes for l in layers)), PinnedBuffer(8 * len(layers))
    pool.fill_random(4, nbytes=pool.nbytes // 8 * 8)
    packed = pool.download()
    words.array[:] = 0
    ctx = TransferContext(0)
    for value in (1, 2):
        ctx.load_layers_marked([l.transfer(b) for l, b in zip(layers, bases(layers, pool.ptr))],
                               [(words.ptr, value, True)], _lib.MODE_KERNEL)
        ctx.synchronize()
        assert words.array.view(np.uint64).tolist() == [value] * len(layers)
        # The first layer; the second; the next three; the last.
        assert ctx.last_stats()[0] == 4
    for l, at in zip(layers, bases(layers, 0)):
        l.restore(packed[at:at + l.nbytes])
        assert np.array_equal(l.dev.download(), l.host)
    ctx.close()


# Chunks around a wave's words and its units at each number of loads per lane,
# a last unit of one word, and launches of one chunk.
FIXED = [(bpb, segs, n) for bpb in (16, 1008, 1024, 1040, 4096, 10240, 16400) for segs, n in
         ((1, 1), (2, 37))]
# The largest call whose descriptors are read in place, and one chunk more.
FIXED += [(1040, 2, 1024), (1040, 1, 2049)]


@pytest.mark.parametrize("bpb,segs,n", FIXED)
def test_fixed_map_copies(gpu, bpb, segs, n):
    """Gather and scatter at every shape of the fixed map, capped grids included."""
    rng = np.random.default_rng(bpb + n)
    (layer,) = make_layers(rng, bpb, segs, (n,), max(64, n + 3))
    pool = DeviceBuffer(layer.nbytes)
    ctx = TransferContext(0)
    shapes = [(t, u | f) for t in (64, 512) for u in (1, 2, 4, 8, 16)
              for f in (0, _lib.KERNEL_NONTEMPORAL, _lib.KERNEL_NT_STORES | _lib.KERNEL_XCD_MAJOR)]
    for i, (threads, unroll) in enumerate(shapes):
        ctx.set_kernel_shape(threads, unroll)
        ctx.set_max_grid((0, 3)[i % 2])
        pool.memset(0)
        ctx.save_layers([layer.transfer(pool.ptr)], _lib.MODE_KERNEL)
        assert np.array_equal(pool.download(), layer.packed()), f"gather {threads} {unroll:#x}"
        pool.fill_random(i, nbytes=pool.nbytes // 8 * 8)
        layer.restore(pool.download())
        ctx.load_layers([layer.transfer(pool.ptr)], _lib.MODE_KERNEL)
        ctx.synchronize()
        assert np.array_equal(layer.dev.download(), layer.host), f"scatter {threads} {unroll:#x}"
    ctx.close()


# Launches of one chunk, of the largest descriptor table read in place and of one
# chunk more, over one layer and over many; whole, partial and tiny tiles.
SMALL = [(bpb, segs, counts) for bpb in (16, 1040, 16400)
         for segs, counts in ((1, (1,)), (2, (3, 0, 1, 4)), (1, (1022, 0, 2)), (1, (1023, 2)),
                              (2, (1,) * 300))]


@pytest.mark.parametrize("bpb,segs,counts", SMALL)
def test_small_host_copies(gpu, bpb, segs, counts):
    """Zero-copy save, load and marked load of few chunks, with one workgroup, a few,
    and more than there are tiles."""
    rng = np.random.default_rng(bpb + len(counts))
    layers = make_layers(rng, bpb, segs, counts, max(counts) + 3)
    pool = PinnedBuffer(sum(l.nbytes for l in layers))
    words = PinnedBuffer(8 * len(layers))
    words.array[:] = 0
    ctx = TransferContext(0)
    xfers = [l.transfer(b) for l, b in zip(layers, bases(layers, pool.ptr))]
    for value, grid in ((1, 1), (2, 3), (3, 64)):
        for route in (_lib.ROUTE_SAVE_HOST, _lib.ROUTE_LOAD_HOST):
            ctx.set_route_grid(route, grid)
        pool.array[:] = 0
        ctx.save_layers(xfers, _lib.MODE_KERNEL)
        assert np.array_equal(pool.array, np.concatenate([l.packed() for l in layers]))
        for marked in (False, True):
            pool.array[:] = rng.integers(0, 256, pool.nbytes, np.uint8)
            if marked:
                ctx.load_layers_marked(xfers, [(words.ptr, value, True)], _lib.MODE_KERNEL)
            else:
                ctx.load_layers(xfers, _lib.MODE_KERNEL)
            ctx.synchronize()
            for l, at in zip(layers, bases(layers, 0)):
                l.restore(pool.array[at:at + l.nbytes])
                assert np.array_equal(l.dev.download(), l.host)
        assert words.array.view(np.uint64).tolist() == [value] * len(layers)
    ctx.close()


# Chunks whose descriptors are read in place, and more than are.
@pytest.mark.parametrize("n", [8, 1100])
def test_more_workgroups_than_tiles(gpu, n):
    """A queue that most workgroups find empty, call after call: save, load and marked
    load, and between device buffers on routes that are set to run queued."""
    (layer,) = make_layers(np.random.default_rng(n), 1040, 1, (n,), n + 3)
    words = PinnedBuffer(8)
    words.array[:] = 0
    ctx = TransferContext(0)
    for route in (_lib.ROUTE_SAVE_HOST, _lib.ROUTE_LOAD_HOST, _lib.ROUTE_SAVE_DEVICE,
                  _lib.ROUTE_LOAD_DEVICE):
        ctx.set_route_grid(route, 5000)
    host, device = PinnedBuffer(layer.nbytes), DeviceBuffer(layer.nbytes)
    for value in (1, 2, 3):
        for pool in (host, device):
            xfer = layer.transfer(pool.ptr)
            ctx.save_layers([xfer], _lib.MODE_KERNEL)
            got = pool.array if pool is host else pool.download()
            assert np.array_equal(got, layer.packed())
            packed = np.random.default_rng(value).integers(0, 256, layer.nbytes, np.uint8)
            if pool is host:
                pool.array[:] = packed
            else:
                pool.upload(packed)
            if pool is host and value == 2:
                ctx.load_layers_marked([xfer], [(words.ptr, value, True)], _lib.MODE_KERNEL)
            else:
                ctx.load_layers([xfer], _lib.MODE_KERNEL)
            ctx.synchronize()
            layer.restore(packed)
            assert np.array_equal(layer.dev.download(), layer.host)
    assert words.array.view(np.uint64).tolist() == [2]
    ctx.close()


# What a call is refused for in its last layer: a block past the tensor, one below it,
# no address for a block, an address in no allocation.
@pytest.mark.parametrize("bad", [("block_idx", 600), ("block_idx", -1), ("k_host", 0),
                                 ("k_host", 4096), ("v_host", 4096)])
def test_refused_device_copy_moves_nothing(gpu, bad):
    """Copies between device buffers of enough chunks to be issued in parts (16 layers of
    512 blocks), with the last layer at fault; without the fault they run."""
    layers = make_layers(np.random.default_rng(5), 256, 2, (512,) * 16, 600)
    pool = DeviceBuffer(sum(l.nbytes for l in layers))
    ctx = TransferContext(0)
    for ok in (False, True):
        xfers = [l.transfer(b) for l, b in zip(layers, bases(layers, pool.ptr))]
        if not ok:
            xfers[-1].blocks[bad[0]][511] = bad[1]
        pool.memset(0xa5)
        if ok:
            ctx.save_layers(xfers, _lib.MODE_KERNEL)
            assert np.array_equal(pool.download(), np.concatenate([l.packed() for l in layers]))
        else:
            with pytest.raises(_lib.PegaFlowError):
                ctx.save_layers(xfers, _lib.MODE_KERNEL)
            assert (pool.download() == 0xa5).all()
        pool.fill_random(7)
        packed = pool.download()
        if ok:
            ctx.load_layers(xfers, _lib.MODE_KERNEL)
        else:
            with pytest.raises(_lib.PegaFlowError):
                ctx.load_layers(xfers, _lib.MODE_KERNEL)
        ctx.synchronize()
        for l, at in zip(layers, bases(layers, 0)):
            if ok:
                l.restore(packed[at:at + l.nbytes])
            assert np.array_equal(l.dev.download(), l.host)
    ctx.close()


# 16 layers, of which the first 4 are a part of their own: the bytes and blocks of those
# and of the others, and whether the others are large enough to be timed.
@pytest.mark.parametrize("first,rest,timed", [((32768, 512), (256, 1024), False),
                                              ((256, 64), (32768, 700), True)])
def test_scatter_trials_time_no_first_part(gpu, first, rest, timed):
    """The scatter's two shapes are compared on launches that are not a call's first part,
    whose share of the call, and so of its fixed costs, is another."""
    rng = np.random.default_rng(3)
    layers = [layer for bpb, n in (first,) * 4 + (rest,) * 12
              for layer in make_layers(rng, bpb, 2, (n,), n + 3)]
    pool = DeviceBuffer(sum(l.nbytes for l in layers))
    pool.fill_random(9)
    packed = pool.download()
    ctx = TransferContext(0)
    for _ in range(4):
        ctx.load_layers([l.transfer(b) for l, b in zip(layers, bases(layers, pool.ptr))],
                        _lib.MODE_KERNEL)
        ctx.synchronize()
    assert ctx.route_shape(_lib.ROUTE_LOAD_DEVICE)[2] is timed
    for l, at in zip(layers, bases(layers, 0)):
        l.restore(packed[at:at + l.nbytes])
        assert np.array_equal(l.dev.download(), l.host)
    ctx.close()


@pytest.mark.parametrize("memory", [PinnedBuffer, DeviceBuffer])
def test_small_calls_one_after_another(gpu, memory):
    """Loads whose descriptors may be read in place, each of its own blocks into its own:
    one behind another with no wait, after a wait, behind marks that were awaited, and
    from two threads that share the context and wait on their own."""
    (layer,) = make_layers(np.random.default_rng(1), 4096, 2, (64,), 6000)
    n, words = 60, PinnedBuffer(8)
    words.array[:] = 0
    ids = np.random.default_rng(2).permutation(6000)[:n * 64].reshape(n, 64)
    pool = memory(n * layer.nbytes)
    packed = np.random.default_rng(3).integers(0, 256, pool.nbytes, np.uint8)
    if memory is PinnedBuffer:
        pool.array[:] = packed
    else:
        pool.upload(packed)
    ctx = TransferContext(0)

    def load(i, marked=False):
        layer.ids = ids[i]
        xfer = [layer.transfer(pool.ptr + i * layer.nbytes)]
        if marked:
            ctx.load_layers_marked(xfer, [(words.ptr, i + 1, True)], _lib.MODE_KERNEL)
            assert host_wait_word(words.ptr, i + 1)
        else:
            ctx.load_layers(xfer, _lib.MODE_KERNEL)

    for i in range(20):
        load(i, marked=i % 5 == 4)
        if i in (3, 9, 10, 16):
            ctx.synchronize()
    lock = threading.Lock()

    def worker(first):
        for i in range(first, n, 2):
            with lock:  # the layer's ids; the wait is outside
                load(i)
            if i % 3 == 0:
                ctx.synchronize()

    threads = [threading.Thread(target=worker, args=(first,)) for first in (20, 21)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    ctx.synchronize()
    for i in range(n):
        layer.ids = ids[i]
        layer.restore(packed[i * layer.nbytes:(i + 1) * layer.nbytes])
    assert np.array_equal(layer.dev.download(), layer.host)
    ctx.close()


# Chunks shorter than a word, around one, around a unit, and of several units, at
# every kind of offset from a word's boundary.
UNALIGNED = [(bpb, off) for bpb in (1, 7, 15, 16, 17, 33, 200, 1009, 1023, 1025, 1041, 2060, 12301)
             for off in (0, 1, 4, 15)]


@pytest.mark.parametrize("bpb,off", UNALIGNED)
def test_unaligned_copies(gpu, bpb, off):
    """Gather and scatter of chunks at odd addresses: every byte of the chunks, and none
    beside them, with and without a capped grid."""
    rng = np.random.default_rng(bpb * 16 + off)
    (layer,) = make_layers(rng, bpb, 2, (23,), 40)
    pool = DeviceBuffer((layer.nbytes + 48) // 8 * 8)
    ctx = TransferContext(0)
    xfer = layer.transfer(pool.ptr + off)
    for cap in (0, 2):
        ctx.set_max_grid(cap)
        pool.memset(0xa5)
        ctx.save_layers([xfer], _lib.MODE_KERNEL)
        got = pool.download()
        assert np.array_equal(got[off:off + layer.nbytes], layer.packed())
        assert (got[:off] == 0xa5).all() and (got[off + layer.nbytes:] == 0xa5).all()
        pool.fill_random(bpb + cap)
        layer.restore(pool.download(layer.nbytes, off))
        ctx.load_layers([xfer], _lib.MODE_KERNEL)
        ctx.synchronize()
        assert np.array_equal(layer.dev.download(), layer.host)
    ctx.close()
