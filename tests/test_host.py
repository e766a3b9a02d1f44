"""Host-side logic of the package that needs no GPU (the reference's unit tests for it)."""

import pytest

from forgeserve_amd import BlockAllocator, ModelConfig, OutOfBlocks, TPContext


def test_config_validation():
    """tests/test_model.py:8-15 of the reference."""
    with pytest.raises(ValueError):
        ModelConfig(d_model=100, n_heads=3)
    with pytest.raises(ValueError):
        ModelConfig(n_heads=8, n_kv_heads=3)
    cfg = ModelConfig(vocab_size=64, d_model=64, n_layers=3, n_heads=8, n_kv_heads=4, max_seq_len=64)
    with pytest.raises(ValueError):
        cfg.check_tensor_parallel(3)
    cfg.check_tensor_parallel(4)
    assert cfg.ffn_dim == 192 and cfg.head_dim == 8
    assert ModelConfig(d_model=256, ffn_dim=688).ffn_dim == 688


def test_allocator():
    """tests/test_paged.py:10-17 of the reference, plus the exact LIFO order."""
    a = BlockAllocator(4)
    got = a.allocate(3)
    assert got == [0, 1, 2] and a.num_free == 1
    with pytest.raises(OutOfBlocks):
        a.allocate(2)
    a.release(got)
    assert a.num_free == 4
    assert a.allocate(2) == [2, 1]


def test_single_gpu_context():
    t = TPContext()
    assert t.size == 1 and t.rank == 0
    with pytest.raises(ValueError):
        TPContext(rank=1, size=1)
    with pytest.raises(NotImplementedError):
        TPContext(rank=0, size=2)


def test_pool_key_layouts():
    """The two key storages of PagedKVPool and the fs_kv_layout each hands the kernels (host only: the
    pool lives on the CPU here and no kernel runs). Grouped keys: a key's 8-dim group g of slot s at
    s * 8 + g * 8 * block_size inside its (block, head) tile; the same element through pool.k."""
    import torch

    from forgeserve_amd import PagedKVPool

    cfg = ModelConfig(vocab_size=32, d_model=256, n_layers=2, n_heads=4, n_kv_heads=2, max_seq_len=64)
    d, bs = cfg.head_dim, 16
    slots = PagedKVPool(cfg, 6, bs, dtype=torch.bfloat16, device="cpu")
    groups = PagedKVPool(cfg, 6, bs, dtype=torch.bfloat16, device="cpu", key_layout="groups")
    ls, lg = slots.layout(1), groups.layout(1)
    assert (ls.k_slot, ls.k_dim, ls.k_group) == (d, 1, 0)
    assert (lg.k_slot, lg.k_dim, lg.k_group) == (8, 1, 8 * bs)
    assert lg.k_block == ls.k_block == 2 * bs * d and lg.k_head == ls.k_head == bs * d
    assert lg.k == groups.k_store[1].data_ptr() and lg.v_dim == ls.v_dim == bs
    assert tuple(groups.k[0].shape) == (6, 2, bs, d // 8, 8)
    # block 3, head 1, slot 5, dim 21 -> group 2, element 5 of it
    groups.k[1][3, 1, 5, 2, 5] = 7.0
    flat = groups.k_store[1].reshape(-1)
    assert float(flat[3 * lg.k_block + 1 * lg.k_head + 5 * lg.k_slot + 2 * lg.k_group + 5]) == 7.0
    assert float(groups.k[1].flatten(-2)[3, 1, 5, 21]) == 7.0
    with pytest.raises(ValueError):
        PagedKVPool(cfg, 6, bs, device="cpu", key_layout="rows")
    with pytest.raises(ValueError):
        PagedKVPool(ModelConfig(vocab_size=32, d_model=48, n_layers=1, n_heads=4, n_kv_heads=2, max_seq_len=16), 4,
                    device="cpu", key_layout="groups")


def test_captures_run_without_the_garbage_collector():
    """Garbage in a reference cycle (as an engine whose method a caller replaced by a closure over it) is
    not collected while a capture is open, whatever the capture's Python allocates; the collector is back
    afterwards, also after nested captures, captures on several threads and an error, and stays off for
    a caller that had it off."""
    import contextlib
    import gc
    import threading

    from forgeserve_amd.speculative import _capturing

    died = []

    class Holder:
        def step(self):
            pass

        def __del__(self):
            died.append(True)

    def garbage():
        h = Holder()
        inner = h.step
        h.step = lambda: inner()   # h -> closure -> bound method -> h

    assert gc.isenabled()
    gc.collect()
    garbage()
    with _capturing(contextlib.nullcontext()):
        with _capturing(contextlib.nullcontext()):
            keep = [[i] for i in range(200_000)]
        keep += [[i] for i in range(200_000)]
        assert not died and not gc.isenabled()
    assert gc.isenabled()
    gc.collect()
    assert died and len(keep) == 400_000

    try:
        with _capturing(contextlib.nullcontext()):
            raise KeyError
    except KeyError:
        pass
    assert gc.isenabled()

    first, second = threading.Event(), threading.Event()

    def other():
        with _capturing(contextlib.nullcontext()):
            first.set()
            second.wait(10)

    t = threading.Thread(target=other)
    t.start()
    first.wait(10)
    with _capturing(contextlib.nullcontext()):
        pass
    assert not gc.isenabled()   # the other thread's capture is still open
    second.set()
    t.join()
    assert gc.isenabled()

    gc.disable()
    try:
        with _capturing(contextlib.nullcontext()):
            pass
        assert not gc.isenabled()
    finally:
        gc.enable()


def _stand_ins(monkeypatch, ran):
    """Native runs of blocks, norms and the two methods of Block and Attention that note what they were asked for
    (there is no GPU here)."""
    from forgeserve_amd import model as mod, ops

    def run_blocks(x, h, b, t, heads, ffn, positions, rope_cos, rope_sin, blocks, normed, buffers):
        ran.append(("run", len(blocks), normed))
        return x, x if normed else None

    monkeypatch.setattr(ops, "add_rmsnorm", lambda x, *a, **kw: x)
    monkeypatch.setattr(ops, "run_blocks", run_blocks)

    def step(self, x, *a, **kw):
        ran.append(("step",))
        return x, x

    monkeypatch.setattr(mod.Block, "step", step)
    monkeypatch.setattr(mod, "_STEP", step)


def _block_model(n_layers, log):
    import torch

    from forgeserve_amd import ForgeModel

    class View:
        def __init__(self, i, log):
            self.i, self.log = i, log

        def prepare(self, b, t, h, d, dtype, device, positions):
            self.log.append(("prepare", self.i))
            return None, None, None, positions

        def commit(self, t):
            self.log.append(("commit", self.i))

    cfg = ModelConfig(vocab_size=8, d_model=32, n_layers=n_layers, n_heads=4, n_kv_heads=2, ffn_dim=64, max_seq_len=16)
    x, pos = torch.zeros(2, 32), torch.zeros(2, 1, dtype=torch.int32)
    model = ForgeModel(cfg)
    views = [View(i, log) for i in range(n_layers)]
    return model, lambda: model._layers(x, 0, n_layers, 2, 1, pos, views, last_norm=model.norm)


@pytest.mark.parametrize("at", [0, 1, 2])
def test_blocks_of_another_kind_run_through_their_step(at, monkeypatch):
    """A layer of another class, without the attributes of Block: every layer runs through its step. A step or attend
    that a caller has replaced on one object, or on the class, is called."""
    import torch

    from forgeserve_amd import model as mod

    ran = []
    _stand_ins(monkeypatch, ran)

    class Foreign(torch.nn.Module):
        attn_norm = torch.nn.Identity()

        def step(self, x, *a, **kw):
            ran.append(("foreign",))
            return x, x

    launches = lambda: [e for e in ran if e[0] not in ("prepare", "commit")]
    model, run = _block_model(3, ran)
    model.layers[at] = Foreign()
    run()
    assert launches() == [("foreign",) if i == at else ("step",) for i in range(3)]

    del ran[:]
    model, run = _block_model(3, ran)   # a step that leaves the norm to the next block
    model.layers[at].step = lambda x, *a, **kw: ran.append(("wrapped",)) or (x, None)
    run()
    assert launches() == [("run", 1, True)] * at + [("wrapped",)] + [("step",)] * (2 - at)

    del ran[:]
    model, run = _block_model(3, ran)
    model.layers[at].attn.attend = lambda *a, **kw: None
    run()
    assert [e[0] for e in launches()].count("step") == (1 if at else 3)   # (the stand-in step does not attend)

    for owner, name in ((mod.Block, "step"), (mod.Attention, "attend")):
        with monkeypatch.context() as m:
            del ran[:]
            model, run = _block_model(3, ran)
            m.setattr(owner, name, lambda self, x, *a, **kw: ran.append(("class",)) or (x, x))
            run()
            assert launches() == [("class",) if name == "step" else ("step",)] * 3


def test_the_first_block_is_launched_before_the_others_are_prepared(monkeypatch):
    """A native run takes one block, then two, four and so on (a last one of one goes with those before it), each
    prepared after the run before it is launched, and committed with its run; a block whose weights are of another dtype takes its step in its place."""
    import torch

    log = []
    _stand_ins(monkeypatch, log)
    for n, runs in ((2, (1, 1)), (4, (1, 3)), (16, (1, 2, 4, 9)), (20, (1, 2, 4, 8, 5))):
        del log[:]
        _block_model(n, log)[1]()
        want, i = [], 0
        for k in runs:
            ids = range(i, i + k)
            want += [("prepare", j) for j in ids] + [("run", k, True)] + [("commit", j) for j in ids]
            i += k
        assert log == want

    del log[:]
    model, run = _block_model(4, log)
    model.layers[2].attn.wo.weight.data = model.layers[2].attn.wo.weight.data.to(torch.bfloat16)
    run()
    assert [e for e in log if e[0] in ("run", "step")] == [("run", 1, True), ("run", 1, True), ("step",), ("run", 1, True)]


def test_a_failed_attention_call_leaves_no_plan_to_reuse(monkeypatch):
    """A call that is refused, by its own checks, for want of memory or by the library, never stands as the one
    whose work plan the next call of the same step reuses; and an earlier one is forgotten only when the
    library has seen the failed call."""
    import os

    import torch

    from forgeserve_amd import ops
    from forgeserve_amd.build import LIB

    if not os.path.exists(LIB):
        pytest.skip("library not built (python -m forgeserve_amd.build)")
    monkeypatch.setattr(ops, "require_device", lambda *a: None)
    monkeypatch.setattr(ops, "stream_ptr", lambda *a: 0)
    monkeypatch.setattr(ops, "_PERSISTENT", {})
    monkeypatch.setattr(ops, "_PLAN_KEY", [None, None])
    key, earlier = object(), object()
    pos, tables = torch.zeros(2, 1, dtype=torch.int32), torch.zeros(2, 1, dtype=torch.int32)
    pool = torch.zeros(2, 2, 16, 8)
    lay = ops.kv_layout(pool, pool)

    def refused(f, error):
        ops._PLAN_KEY[:] = earlier, pos
        with pytest.raises(error):
            f()
        assert ops._PLAN_KEY[0] is not key
        return ops._PLAN_KEY[0]

    # three query heads over two KV heads: the library refuses them
    three = lambda f, q, *a: refused(lambda: f(q, lay, tables, pos, *a, 1.0, plan_key=key), ValueError)
    assert three(ops.paged_attention, torch.zeros(2, 1, 3, 8)) is None
    assert three(ops.paged_attention_varlen, torch.zeros(2, 3, 8), torch.tensor([0, 1, 2], dtype=torch.int32)) is None

    x, w = torch.zeros(2, 32), torch.zeros(64, 32)
    block = lambda tab: (w, w, w, w, x[0], 1e-5, x[0], 1e-5, (lay, tab, None, pos), key)
    run = lambda blocks: ops.run_blocks(x, x, 2, 1, (4, 2, 8), 32, pos, x, x, blocks, True, {})
    assert refused(lambda: run([block(tables), block(tables.long())]), ValueError) is earlier

    def full(*a):
        raise torch.OutOfMemoryError("none left")

    monkeypatch.setattr(ops, "_ws", full)
    assert refused(lambda: run([block(tables)]), torch.OutOfMemoryError) is earlier
