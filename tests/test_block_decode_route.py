"""CPU-only checks of which decode steps of a block go to the native call: a block of plain modules does, and whatever a
caller has put in the way of the general step keeps that step.  The native module is replaced by a recorder."""
import pytest
import torch
from torch.overrides import TorchFunctionMode
from torch.utils.flop_counter import FlopCounterMode

from energonai_amd import _lib
from energonai_amd.kernel import LayerNorm
from energonai_amd.model import MLP1D, Block1D, MultiHeadAttention1D
from energonai_amd.model.kv_cache import KVCache, OutputHistory


class Recorder:
    def __init__(self):
        self.calls = []

    def block_decode(self, *args):
        self.calls.append(args)
        return args[0]


@pytest.fixture
def step(monkeypatch):
    """A block behind its prompt of 8 positions, and a function that runs one decode step's choice of route."""
    front = Recorder()
    monkeypatch.setattr(_lib, "front", front)
    blk = Block1D(128, 2, 2.0, activation=torch.nn.GELU(), dtype=torch.float16, max_seq_len=32)
    blk.attn.kv_cache = KVCache(2, 2, 32, 64, torch.float16, "cpu")
    blk._history.start(torch.zeros(2, 8, 128, dtype=torch.float16), 32)

    def run():
        del front.calls[:]
        with torch.no_grad():
            blk._native_decode(torch.zeros(2, 1, 128, dtype=torch.float16))
        return bool(front.calls)

    return blk, run


def test_a_block_of_plain_modules_takes_the_native_call(step, monkeypatch):
    blk, run = step
    assert run() and blk._history.cur == 9 and blk.attn.kv_cache._longest == 1
    with torch.device("cpu"):           # a default device alone changes nothing
        assert run()


def test_the_limits_are_the_entry_points(step):
    """The look that spares a call is at the limits of the header, so that neither side can move alone."""
    import os
    import re
    from energonai_amd import build
    from energonai_amd.model import endecoder
    with open(os.path.join(build.INCLUDE, "energon_hip.h")) as f:
        defines = dict(re.findall(r"#define EN_BLOCK_DECODE_MAX_(\w+) (\d+)", f.read()))
    assert defines == {"BATCH": str(endecoder.NATIVE_MAX_BATCH), "HIDDEN": str(endecoder.NATIVE_MAX_HIDDEN)}


@pytest.mark.parametrize("what", ["float32", "batch", "hidden", "activation", "post_layernorm"])
def test_blocks_without_a_kernel_are_seen_before_their_modules_are_gone_through(step, monkeypatch, what):
    """They stay with the general step, and what its look costs them is that of a few attributes."""
    from energonai_amd.model import endecoder
    blk, _ = step
    looked = []
    monkeypatch.setattr(endecoder, "_step_methods", lambda: looked.append(1))
    x = torch.zeros((33 if what == "batch" else 2, 1, 2304 if what == "hidden" else 128),
                    dtype=torch.float32 if what == "float32" else torch.float16)
    if what == "activation":
        blk.mlp.activation = torch.nn.SiLU()
    blk.apply_post_layernorm = what == "post_layernorm"
    with torch.no_grad():
        assert blk._native_decode(x) is None
    assert not looked and not _lib.front.calls and blk._history.cur == 8


def _plain_attribute(name):
    def change(module):
        value = getattr(module, name).detach().clone()
        delattr(module, name)
        setattr(module, name, value)
    return change


class OwnCache(KVCache):
    def attend(self, q, scale):
        return super().attend(q, scale)


class DuckCache:
    """Only what the general step asks of a cache."""

    def append(self, k, v):
        pass

    def attend(self, q, scale):
        return q

    _longest = 0


class OwnHistory(OutputHistory):
    def push(self, new):
        return super().push(new)


def _own_history(blk):
    blk._history.__class__ = OwnHistory


def _on_instance(path, name):
    """Sets the module's method again on the instance, as an instrumenting caller does."""
    def change(blk):
        obj = blk
        for part in path.split(".") if path else ():
            obj = getattr(obj, part)
        method = getattr(obj, name)
        obj.__dict__[name] = lambda *args, **kwargs: method(*args, **kwargs)
    return change


CHANGES = {
    "rows_on_instance": _on_instance("", "_rows"),
    "forward_last_on_instance": _on_instance("attn", "forward_last"),
    "project_on_instance": _on_instance("attn", "_project"),
    "forward_rows_on_instance": _on_instance("mlp", "forward_rows"),
    "norm1_forward_on_instance": _on_instance("norm1", "forward"),
    "norm2_forward_on_instance": _on_instance("norm2", "forward"),
    "qkv_forward_on_instance": _on_instance("attn.query_key_value", "forward"),
    "dense_forward_on_instance": _on_instance("attn.dense", "forward"),
    "fc1_forward_on_instance": _on_instance("mlp.dense_1", "forward"),
    "fc2_forward_on_instance": _on_instance("mlp.dense_2", "forward"),
    "activation_forward_on_instance": _on_instance("mlp.activation", "forward"),
    "cache_append_on_instance": _on_instance("attn.kv_cache", "append"),
    "history_push_on_instance": _on_instance("_history", "push"),
    "cache_subclass": lambda blk: setattr(blk.attn.kv_cache, "__class__", OwnCache),
    "cache_of_another_class": lambda blk: setattr(blk.attn, "kv_cache", DuckCache()),
    "history_subclass": _own_history,
    "compiled_module": lambda blk: setattr(blk.mlp.dense_1, "_compiled_call_impl", blk.mlp.dense_1._call_impl),
    "weight_as_plain_attribute": lambda blk: _plain_attribute("weight")(blk.attn.dense),
    "bias_as_plain_attribute": lambda blk: _plain_attribute("bias")(blk.mlp.dense_1),
    "norm_weight_as_plain_attribute": lambda blk: _plain_attribute("weight")(blk.norm2),
    "weight_as_buffer": lambda blk: (blk.mlp.dense_2.__delattr__("weight"),
                                     blk.mlp.dense_2.register_buffer("weight", torch.zeros(128, 256, dtype=torch.float16))),
    "module_as_plain_attribute": lambda blk: (lambda mlp: (blk.__delattr__("mlp"), blk.__dict__.__setitem__("mlp", mlp)))(blk.mlp),
}


@pytest.mark.parametrize("name", list(CHANGES))
def test_what_a_caller_put_in_keeps_the_general_step(step, name):
    blk, run = step
    CHANGES[name](blk)
    assert not run()
    assert blk._history.cur == 8 and blk.attn.kv_cache._longest == 0


@pytest.mark.parametrize("owner,name", [(Block1D, "_rows"), (MultiHeadAttention1D, "forward_last"), (MultiHeadAttention1D, "_project"),
                                        (MLP1D, "forward_rows"), (LayerNorm, "forward"), (torch.nn.Linear, "forward"), (torch.nn.functional, "linear"),
                                        (torch.nn.GELU, "forward"), (torch.nn.functional, "gelu"),
                                        (OutputHistory, "push"), (KVCache, "append"), (KVCache, "attend")])
def test_methods_replaced_on_the_class_keep_the_general_step(step, monkeypatch, owner, name):
    blk, run = step
    method = getattr(owner, name)
    monkeypatch.setattr(owner, name, lambda *args, **kwargs: method(*args, **kwargs))
    assert not run()
    assert blk._history.cur == 8 and blk.attn.kv_cache._longest == 0


class Passing(TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("mode", [Passing, lambda: FlopCounterMode(display=False)])
def test_modes_that_watch_the_projections_keep_the_general_step(step, mode):
    blk, run = step
    with mode():
        assert not run()
    assert run()


@pytest.fixture
def prefill(monkeypatch):
    """A block and a function that runs one prefill's choice of route on packed rows that claim to be on the GPU."""
    from energonai_amd.model import endecoder
    from energonai_amd.seqinfo import SeqInfo

    class Rows(torch.Tensor):
        is_cuda = True

    calls = []

    class Front:
        def prefix_sum(self, lens, batch):
            return torch.cat((lens.new_zeros(1), lens.cumsum(0).int())), lens

        def block_prefill(self, *args):
            calls.append(args)
            return None

    monkeypatch.setattr(_lib, "front", Front())
    monkeypatch.setattr(endecoder, "linear_entry", lambda device: (1, None))
    blk = Block1D(128, 2, 2.0, activation=torch.nn.GELU(approximate="tanh"), dtype=torch.float16, max_seq_len=32)
    lens = torch.tensor([3, 5], dtype=torch.int32)
    batch = SeqInfo(lens, lens, 2, 8, None)
    batch.ephemeral = True

    def run(fill=True, S=8, info=batch, batch_size=2):
        del calls[:]
        with torch.no_grad():
            assert blk._native_prefill(torch.zeros(1, 8, 128, dtype=torch.float16).as_subclass(Rows), info, batch_size, S, fill) is None
        return bool(calls)

    return blk, run


def test_a_prefill_of_plain_modules_takes_the_native_call(prefill):
    blk, run = prefill
    assert run() and run(fill=False)
    assert not run(S=33) and run(fill=False, S=33)        # longer than the cache: the general form says so


def test_a_native_prefill_waits_for_the_lengths(prefill, monkeypatch):
    """The prefix sum may have been launched on another stream; a SeqInfo without a tile table is waited for as well."""
    from energonai_amd.seqinfo import SeqInfo
    blk, run = prefill
    events = []
    monkeypatch.setattr(SeqInfo, "order_current_stream", lambda self: events.append("ordered"))
    native = _lib.front.block_prefill
    monkeypatch.setattr(_lib.front, "block_prefill", lambda *args: events.append("launched") or native(*args), raising=False)
    assert run() and events[0] == "ordered" and events.count("launched") == 1 and events[-1] == "launched"


@pytest.mark.parametrize("batch_size", [1, 3])
def test_a_native_prefill_refuses_lengths_of_another_batch(prefill, batch_size):
    blk, run = prefill
    with pytest.raises(RuntimeError, match="SeqInfo was built for batch 2"):
        run(batch_size=batch_size)
    assert blk.attn.kv_cache is None


def test_a_native_prefill_takes_plain_lengths(prefill):
    """Lengths that are not a SeqInfo become one, as in the general form's attention."""
    blk, run = prefill
    assert run(info=[3, 5], fill=False)


@pytest.mark.parametrize("page", [None, 16])
def test_a_cache_that_could_not_be_filled_is_not_kept(monkeypatch, page):
    """Its rows and lengths are uninitialised memory: the module keeps the cache it had."""
    from energonai_amd.model.kv_cache import PagedKVCache

    def fail(self, *args, **kwargs):
        raise RuntimeError("not filled")

    for cache in (KVCache, PagedKVCache):
        monkeypatch.setattr(cache, "fill", fail)
    attn = MultiHeadAttention1D(128, 2, max_seq_len=32, kv_page_size=page)
    kvq = torch.zeros(8, 6, 64, dtype=torch.float16)
    for before in (None, KVCache(2, 2, 32, 64, torch.float16, "cpu")):
        attn.kv_cache = before
        with pytest.raises(RuntimeError, match="not filled"):
            attn._start_cache(None, None, kvq, None, 2, 8)
        assert attn.kv_cache is before


class DuckHistory:
    """Only what a module asks of a history."""
    __slots__ = ("got",)

    def start(self, out, max_seq_len):
        self.got = (out, max_seq_len)
        return out

    def push(self, new):
        return new


class StartsByItself(OutputHistory):
    def start(self, out, max_seq_len):
        self.got = (out, max_seq_len)
        return out


def test_a_history_of_the_callers_own_is_started_with_padded_rows(monkeypatch):
    """Whatever has ``start`` and ``push``; the package's own takes the packed rows."""
    from energonai_amd.model import attention, endecoder, kv_cache, stack
    assert attention.start_history is endecoder.start_history is stack.start_history is kv_cache.start_history
    packed, padded = torch.ones(1, 8, 128), torch.zeros(2, 8, 128)
    monkeypatch.setattr(kv_cache, "repad", lambda y, *args, out=None, **kwargs: padded if out is None else out)
    on_instance = OutputHistory()
    on_instance.start = lambda out, max_seq_len: setattr(on_instance, "got", (out, max_seq_len)) or out
    for history in (DuckHistory(), StartsByItself(), on_instance):
        assert kv_cache.start_history(history, packed, 2, 8, None, False, 32) is padded and history.got == (padded, 32)
    own = OutputHistory()
    assert kv_cache.start_history(own, packed, 2, 8, None, False, 32).shape == (2, 8, 128) and own.buf.shape == (2, 32, 128) and own.cur == 8


def test_a_cache_saved_before_it_could_be_unzeroed_is_filled(monkeypatch):
    """A pickled cache of that time has zeros in its buffers and says nothing about them."""
    from energonai_amd.model import kv_cache
    from energonai_amd.seqinfo import SeqInfo
    filled = []
    monkeypatch.setattr(kv_cache, "kv_cache_fill", lambda *args, zero_padding: filled.append(zero_padding))
    monkeypatch.setattr(kv_cache, "kv_cache_start", lambda *args: filled.append("start"))
    cache = KVCache(2, 2, 32, 64, torch.float16, "cpu")
    del cache.__dict__["_zeroed"]
    lens, rows = torch.tensor([3, 5], dtype=torch.int32), torch.zeros(8, 6, 64, dtype=torch.float16)
    cache.fill(rows, rows, SeqInfo(lens, lens, 2, 8, None), 0, 2)
    assert filled == [False, False] and cache.lens.tolist() == [3, 5]


PREFILL_CHANGES = {name: CHANGES[name] for name in CHANGES
                   if "cache" not in name and "history" not in name and "activation" not in name and "forward_last" not in name}
PREFILL_CHANGES.update({
    "forward_packed_on_instance": _on_instance("attn", "forward_packed"),
    "start_cache_on_instance": _on_instance("attn", "_start_cache"),
    "post_layernorm": lambda blk: setattr(blk, "apply_post_layernorm", True),
    "other_activation": lambda blk: setattr(blk.mlp, "activation", torch.nn.SiLU()) or setattr(blk.mlp, "_epilogue", None),
    "heads_that_the_projections_do_not_have": lambda blk: setattr(blk.attn, "num_heads", 4),
    "separate_projections": lambda blk: setattr(blk.attn, "fused_qkv", False),
})


@pytest.mark.parametrize("name", list(PREFILL_CHANGES))
def test_what_a_caller_put_in_keeps_the_general_prefill(prefill, name):
    blk, run = prefill
    PREFILL_CHANGES[name](blk)
    assert not run()


@pytest.mark.parametrize("owner,name", [(Block1D, "_rows"), (MultiHeadAttention1D, "forward_packed"), (MultiHeadAttention1D, "_project"),
                                        (MLP1D, "forward_rows"), (LayerNorm, "forward"), (torch.nn.Linear, "forward"),
                                        (torch.nn.functional, "linear"), (torch.nn.functional, "gelu")])
def test_methods_replaced_on_the_class_keep_the_general_prefill(prefill, monkeypatch, owner, name):
    blk, run = prefill
    method = getattr(owner, name)
    monkeypatch.setattr(owner, name, lambda *args, **kwargs: method(*args, **kwargs))
    assert not run()


@pytest.mark.parametrize("mode", [Passing, lambda: FlopCounterMode(display=False)])
def test_modes_that_watch_the_projections_keep_the_general_prefill(prefill, mode):
    blk, run = prefill
    with mode():
        assert not run()
    assert run()
