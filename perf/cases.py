"""The transfer path's work, case by case, through its public entry points.

A case is one transfer call as a serving worker makes it: the KV blocks of one
request moved between a model's paged KV tensors in HBM and the place that keeps
them, a pinned host pool or a buffer in HBM.  The tensors are torch's, as a model
runner allocates them; the pinned memory, the transfer context, the engine and the
block lists are what such a worker holds before the call.

``op`` of a case:
  * ``save``     TransferContext.save_layers: paged blocks -> pool (returns with the
                 bytes in place);
  * ``load``     TransferContext.load_layers and a synchronize: pool -> paged blocks;
  * ``layered``  TransferContext.load_layers_marked, waiting for each layer's word in
                 layer order, as a layer-by-layer forward pass does;
  * ``engine``   PegaEngine.batch_load_kv_blocks by hash with a layered LoadState,
                 polled until it reads ready.
"""

import numpy as np
import torch

from pegaflow_amd import _lib
from pegaflow_amd.engine import PegaEngine
from pegaflow_amd.load_state import PyLoadState
from pegaflow_amd.runtime import PinnedBuffer, host_wait_word
from pegaflow_amd.transfer import BLOCK_DTYPE, KVCacheRegistration, LayerTransfer, TransferContext
from pegaflow_amd.workload import save_plan

KIB, MIB, GIB = 1 << 10, 1 << 20, 1 << 30
MODES = {"auto": _lib.MODE_AUTO, "kernel": _lib.MODE_KERNEL}
# Staging of a transfer context whose host copies may run on the copy engines: what
# the engine gives its save and load contexts.
STAGING = 512 * MIB
MAX_PAYLOAD = 1280 * MIB
MAX_TENSORS = 39 * GIB


def _case(name, op, layers, num_blocks, block_bytes, segments, blocks, *, pool="host",
          mode="auto", run=1, batch=0):
    """layers x [segments, num_blocks, block_bytes] tensors, of which ``blocks`` blocks
    move.  ``run``: the paged blocks come in runs of so many neighbours.  ``batch``: the
    pool holds them in saved batches of so many blocks (0: one batch)."""
    c = {"op": op, "pool": pool, "mode": mode, "layers": layers, "num_blocks": num_blocks,
         "block_bytes": block_bytes, "segments": segments, "blocks": blocks, "run": run,
         "batch": batch}
    return {"name": name, **c} if name else c


def listed():
    return [
        # The smallest call: one block of 16 tokens x 32 layers comes back for a request
        # whose prefix grew by one block (2 MiB; [2, 20000, 16, 8, 128] in bf16).
        _case("load_1_block", "load", 32, 20000, 32 * KIB, 2, 1),
        # A decode step's saves: the blocks that five requests filled in this step.
        _case("save_5_blocks", "save", 32, 20000, 32 * KIB, 2, 5),
        # A short prompt's prefix by hash through the engine, layer by layer.
        _case("engine_load_16_blocks", "engine", 32, 2000, 32 * KIB, 2, 16),
        # A multi-turn prefix: 77 blocks saved 8 at a time by earlier steps, 24 KiB
        # segments (12 layers of [2, 512, 16, 12, 64] in fp16).
        _case("load_77_blocks_batched", "load", 12, 512, 24 * KIB, 2, 77, batch=8),
        # A layout whose blocks are no multiple of 16 bytes (packed quantized values
        # with their scales): every address of the copy is odd-sized.
        _case("load_ragged_blocks", "load", 24, 1000, 12300, 2, 100),
        # One tensor-parallel rank's shard: 4 KiB segments, a 10,000-token prompt saved.
        _case("save_4kib_segments", "save", 32, 20000, 4 * KIB, 2, 640),
        # A latent cache in 8 bits, one segment a block ([8192, 64, 576]), handed over in
        # an HBM buffer and put in place layer by layer.
        _case("layered_latent_from_hbm", "layered", 61, 8192, 36 * KIB, 1, 128, pool="hbm",
              mode="kernel"),
        # A 5,000-token prompt restored layer by layer under a forward pass.
        _case("layered_313_blocks", "layered", 36, 4000, 32 * KIB, 2, 313),
        # The 10,000-token prompt: saved, restored, and moved to and from an HBM buffer.
        _case("save_640_blocks", "save", 32, 4000, 32 * KIB, 2, 640),
        _case("load_640_blocks", "load", 32, 4000, 32 * KIB, 2, 640, mode="kernel"),
        _case("gather_640_blocks_hbm", "save", 32, 20000, 32 * KIB, 2, 640, pool="hbm",
              mode="kernel"),
        _case("scatter_640_blocks_hbm", "load", 32, 20000, 32 * KIB, 2, 640, pool="hbm",
              mode="kernel"),
    ]


def draw(rng):
    """Any of the calls above over their whole range: 1 to 1024 blocks of 1 to 128 KiB in
    4 to 64 layers, up to the payload of the largest listed case."""
    op = rng.choice(("load", "load", "save", "save", "layered", "engine"))
    pool = "host" if op == "engine" else rng.choice(("host", "host", "hbm"))
    mode = "kernel" if pool == "hbm" or rng.random() < 0.25 else "auto"
    layers = rng.randint(4, 64)
    if rng.random() < 0.25:  # a latent cache: one segment a block
        segments, block_bytes = 1, rng.choice((16, 32, 64)) * 576 * rng.choice((1, 2))
    else:
        segments = 2
        block_bytes = 16 * rng.randint(1, 8) * rng.choice((64, 80, 96, 128, 192)) * rng.choice((1, 2))
    if rng.random() < 0.15:
        block_bytes += rng.randint(1, 15)
    per_block = layers * segments * block_bytes
    most = max(1, min(1024, MAX_PAYLOAD // per_block))
    blocks = max(1, min(most, round(most ** rng.random())))
    num_blocks = max(blocks + 8, min(round(blocks * 2 ** rng.uniform(1, 6)), 20000,
                                     MAX_TENSORS // per_block))
    return _case(None, op, layers, num_blocks, block_bytes, segments, blocks, pool=pool,
                 mode=mode, run=rng.choice((1, 1, 4, 32)),
                 batch=rng.choice((0, 0, 0, 8, 64)) if op == "load" else 0)


class _PinnedWords:
    """A pinned buffer as an array that keeps the buffer: what a case returns may be
    read after its state is gone."""

    def __init__(self, nbytes):
        self.buffer = PinnedBuffer(nbytes)
        self.ptr = self.buffer.ptr
        self.__array_interface__ = self.buffer.array.view(np.int64).__array_interface__


def _payload(c):
    return c["layers"] * c["segments"] * c["block_bytes"] * c["blocks"]


def _tensors(c, generator):
    """All layers' KV tensors in one torch allocation, padded to 256 bytes a layer, and
    their registrations.  A save reads seeded values; a load finds zeros."""
    stride = c["num_blocks"] * c["block_bytes"]
    size = stride * c["segments"]
    words = (size + 255) // 256 * 32
    kv = torch.empty((c["layers"], words), dtype=torch.int64, device="cuda")
    if c["op"] == "save":
        kv.random_(generator=generator)
    else:
        kv.zero_()
    regs = [KVCacheRegistration.create(kv[i].data_ptr(), size, c["num_blocks"], c["block_bytes"],
                                       stride if c["segments"] == 2 else 0, c["segments"])
            for i in range(c["layers"])]
    return kv, regs


def _block_ids(c, seed):
    """Distinct blocks in the order of the request, in runs of c["run"] neighbours."""
    rng = np.random.default_rng(seed)
    run = min(c["run"], c["num_blocks"] // c["blocks"]) or 1
    starts = rng.permutation(c["num_blocks"] // run)[:-(-c["blocks"] // run)]
    return (starts[:, None] * run + np.arange(run)).reshape(-1)[:c["blocks"]].astype(np.int64)


def _transfers(c, regs, ids, base):
    """The call's block lists: each saved batch in the pool's layout (a K and a V region
    a layer, or one of whole blocks), one batch after another from ``base``."""
    step = c["batch"] or len(ids)
    batches = []
    for i in range(0, len(ids), step):
        batches.append(save_plan(regs, ids[i:i + step], base))
        base += sum(r.block_size_bytes for r in regs) * len(ids[i:i + step])
    return [LayerTransfer(reg, np.concatenate([b[l].blocks for b in batches]).astype(BLOCK_DTYPE))
            for l, reg in enumerate(regs)]


def _prepare_engine(c, kv, regs, ids, generator):
    """An engine that holds the request's blocks, saved from other blocks' values."""
    engine = PegaEngine(pool_size=_payload(c) + 64 * MIB)
    names = ["layer.%d" % i for i in range(c["layers"])]
    for name, r in zip(names, regs):
        engine.register_context_layer("instance", "namespace", 0, name, r.data_ptr, r.size_bytes,
                                      r.num_blocks, r.bytes_per_block, r.kv_stride_bytes,
                                      r.segments, 0, 1, c["layers"])
    hashes = [b"block %d" % i for i in range(len(ids))]
    kv.random_(generator=generator)
    torch.cuda.synchronize()
    engine.batch_save_kv_blocks("instance", 0, 0, [(n, ids.tolist(), hashes) for n in names])
    kv.zero_()
    targets = _block_ids(c, int(ids.sum()) + 1)
    return {"op": "engine", "engine": engine, "names": names, "hashes": hashes,
            "ids": targets.tolist(), "kv": kv, "layers": c["layers"]}


def prepare(case, seed):
    c = case
    generator = torch.Generator(device="cuda")
    generator.manual_seed(seed)
    kv, regs = _tensors(c, generator)
    ids = _block_ids(c, seed)
    if c["op"] == "engine":
        state = _prepare_engine(c, kv, regs, ids, generator)
        torch.cuda.synchronize()
        return state
    ctx = TransferContext(0, staging_bytes=STAGING if c["mode"] == "auto" else 0)
    words = (_payload(c) + 7) // 8
    if c["pool"] == "host":
        pinned = _PinnedWords(words * 8)
        pool, base = np.asarray(pinned), pinned.ptr
        if c["op"] == "save":
            pool[:] = 0
        else:
            values = torch.empty(words, dtype=torch.int64, device="cuda")
            values.random_(generator=generator)
            torch.from_numpy(pool).copy_(values)
    else:
        pool = torch.zeros(words, dtype=torch.int64, device="cuda")
        base = pool.data_ptr()
        if c["op"] != "save":
            pool.random_(generator=generator)
    state = {"op": c["op"], "ctx": ctx, "mode": MODES[c["mode"]], "pool": pool, "kv": kv,
             "transfers": _transfers(c, regs, ids, base)}
    if c["op"] == "layered":
        state["words"] = PinnedBuffer(8 * c["layers"])
        state["words"].array[:] = 0
        state["passes"] = 0
    torch.cuda.synchronize()
    return state


def run(state):
    op = state["op"]
    if op == "engine":
        done = PyLoadState(num_layers=state["layers"])
        state["engine"].batch_load_kv_blocks("instance", 0, 0, done.shm_name(), state["names"],
                                             state["ids"], state["hashes"])
        while not done.is_ready():
            pass
        if done.get_state() < 0:
            raise RuntimeError("the engine's load failed")
        return state["kv"]
    ctx, transfers = state["ctx"], state["transfers"]
    if op == "save":
        ctx.save_layers(transfers, state["mode"])
        return state["pool"]
    if op == "load":
        ctx.load_layers(transfers, state["mode"])
        ctx.synchronize()
        return state["kv"]
    state["passes"] += 1
    word = state["words"].ptr
    ctx.load_layers_marked(transfers, [(word, state["passes"], True)], state["mode"])
    for i in range(len(transfers)):
        if not host_wait_word(word + 8 * i, state["passes"]):
            raise RuntimeError("a layer's word never came")
    return state["kv"]


def work(case):
    """Each byte of the blocks read once where it lies and written once where it goes."""
    return {"bytes": 2 * _payload(case), "flops": 0}


def tolerance(case):
    return "exact"  # bytes move; none is computed
