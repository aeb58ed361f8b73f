"""Which prefills write K/V in the launch that rotates them, and which go
through the caller's own qk_norm_rope, forward and store_kv (CPU only)."""
from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch

from aios_amd import _lib
from aios_amd.attention.backend import Mi355xAttentionBackend, Mi355xAttentionMetadata
from aios_amd.kvcache import MHAKVCache
from aios_amd.layers import HipOps
from aios_amd.qwen3 import Qwen3ForCausalLM

CFG = SimpleNamespace(num_qo_heads=4, num_kv_heads=2, head_dim=64, rms_norm_eps=1e-6)


class _GpuTensor(torch.Tensor):
    is_cuda = True


def _pool(cls=MHAKVCache, dtype=torch.bfloat16, heads=2):
    p = cls.__new__(cls)
    p._kv_buffer = torch.empty(2, 1, 8, 1, heads, 64, dtype=dtype)
    p._storage_shape = (8, heads, 64)
    return p


def _batch(loc=None, tokens=3, phase="prefill", total_q=3):
    md = object.__new__(Mi355xAttentionMetadata)
    md.plan = _lib.AttnPlan()
    md.plan.total_q = total_q
    loc = torch.zeros(tokens, dtype=torch.int32).as_subclass(_GpuTensor) if loc is None else loc
    return SimpleNamespace(is_prefill=phase == "prefill", is_decode=phase != "prefill",
                           out_loc=loc, attn_metadata=md, fused_append=False)


class _OwnStore(MHAKVCache):
    def store_kv(self, k, v, out_loc, layer_id):
        return super().store_kv(k, v, out_loc, layer_id)


class _OwnCaches(MHAKVCache):
    def k_cache(self, index):
        return super().k_cache(index)


class _PlainSubclass(MHAKVCache):
    pass


class _Proxy:
    """A pool that forwards what it does not have itself."""

    def __init__(self, pool):
        self.pool = pool

    def __getattr__(self, name):
        return getattr(self.pool, name)


class _SlottedProxy:
    __slots__ = ("pool",)

    def __init__(self, pool):
        self.pool = pool

    def __getattr__(self, name):
        return getattr(self.pool, name)


class _OwnForward(Mi355xAttentionBackend):
    def forward(self, q, k, v, paged_kv_cache, layer_id, batch):
        return super().forward(q, k, v, paged_kv_cache, layer_id, batch)


def _with(obj, **attrs):
    for k, v in attrs.items():
        setattr(obj, k, v)
    return obj


BF = torch.bfloat16
I64 = torch.zeros(3, dtype=torch.int64).as_subclass(_GpuTensor)
GAPS = torch.zeros(6, dtype=torch.int32).as_subclass(_GpuTensor)[::2]


@pytest.mark.parametrize("backend,pool,batch,rows,taken", [
    (Mi355xAttentionBackend(CFG), _pool(), _batch(), 3, True),
    (Mi355xAttentionBackend(CFG), _pool(_PlainSubclass), _batch(), 3, True),
    (Mi355xAttentionBackend(CFG), _pool(), _batch(phase="decode"), 3, False),
    (Mi355xAttentionBackend(CFG), _pool(), _batch(loc=I64), 3, False),
    (Mi355xAttentionBackend(CFG), _pool(), _batch(loc=GAPS), 3, False),
    (Mi355xAttentionBackend(CFG), _pool(), _batch(loc=torch.zeros(3, dtype=torch.int32)), 3, False),
    (Mi355xAttentionBackend(CFG), _pool(), _batch(tokens=4), 3, False),
    (Mi355xAttentionBackend(CFG), _pool(), _batch(total_q=4), 3, False),
    (Mi355xAttentionBackend(CFG), _pool(), _batch(), 4, False),
    (Mi355xAttentionBackend(CFG), _pool(dtype=torch.float16), _batch(), 3, False),
    (Mi355xAttentionBackend(CFG), _pool(heads=4), _batch(), 3, False),
    (Mi355xAttentionBackend(CFG), _pool(_OwnStore), _batch(), 3, False),
    (Mi355xAttentionBackend(CFG), _pool(_OwnCaches), _batch(), 3, False),
    (Mi355xAttentionBackend(CFG), _with(_pool(), store_kv=lambda *a: None), _batch(), 3, False),
    (Mi355xAttentionBackend(CFG), _Proxy(_pool()), _batch(), 3, False),
    (Mi355xAttentionBackend(CFG), _SlottedProxy(_pool()), _batch(), 3, False),
    (_OwnForward(CFG), _pool(), _batch(), 3, False),
    (_with(Mi355xAttentionBackend(CFG), forward=lambda *a: None), _pool(), _batch(), 3, False),
])
def test_append_rope_applies(backend, pool, batch, rows, taken):
    qkv = torch.zeros(rows, 8 * 64, dtype=BF)
    assert backend.append_rope_applies(qkv, pool, batch) is taken


def test_a_wrapped_store_of_the_class_is_called(monkeypatch):
    """store_kv replaced on the class itself (a hook of the caller's)."""
    be = Mi355xAttentionBackend(CFG)
    args = (torch.zeros(3, 8 * 64, dtype=BF), _pool(), _batch())
    assert be.append_rope_applies(*args)
    monkeypatch.setattr(MHAKVCache, "store_kv", lambda self, *a: None)
    assert not be.append_rope_applies(*args)


class _OwnRope(HipOps):
    @staticmethod
    def qk_norm_rope(*args):
        return HipOps.qk_norm_rope(*args)


class _Forwarding:
    """An op set or backend that wraps another one."""

    def __init__(self, inner, log):
        self.inner, self.log = inner, log

    def __getattr__(self, name):
        return getattr(self.inner, name)

    def qk_norm_rope(self, *args):
        self.log.append("own rope")
        return self.inner.qk_norm_rope(*args)

    def forward(self, *args):
        self.log.append("own forward")
        return self.inner.forward(*args)


@pytest.mark.parametrize("kind", ["plain", "ops subclass", "ops attribute", "ops wrapper",
                                  "backend wrapper"])
def test_own_ops_and_backends_see_every_prefill(kind):
    """attention_core takes the one-launch form only past no call of the caller's own."""
    log = []

    def call(name, out=None):
        return lambda *a, **k: log.append(name) or out

    be = _with(Mi355xAttentionBackend(CFG), append_rope_applies=lambda *a: True,
               layer_kv=call("layer_kv", (None, None)), prefill_appended=call("appended"),
               forward=call("forward"))
    ops = _OwnRope() if kind == "ops subclass" else HipOps()
    ops.qk_norm_rope_append = call("append")
    if kind == "ops attribute":
        ops.qk_norm_rope = call("rope", (None, None))
    elif kind == "ops subclass":
        _OwnRope.qk_norm_rope = staticmethod(call("rope", (None, None)))
    elif kind == "ops wrapper":
        ops = _Forwarding(ops, log)
        ops.inner = SimpleNamespace(rope_in_append=True, qk_norm_rope=call("rope", (None, None)),
                                    qk_norm_rope_append=call("append"))
    elif kind == "backend wrapper":
        ops = _with(HipOps(), qk_norm_rope_append=call("append"))
    model = Qwen3ForCausalLM.__new__(Qwen3ForCausalLM)
    model.config, model.ops = CFG, ops
    model.attn_backend = _Forwarding(be, log) if kind == "backend wrapper" else be
    model.w = {"layers": [{"q_norm": None, "k_norm": None}]}
    model.rotary = SimpleNamespace(cos=None, sin=None)
    model._q_size, model._kv_size = 4 * 64, 2 * 64
    qkv = torch.zeros(3, 8 * 64, dtype=BF)
    if kind == "backend wrapper":
        # the wrapper's forward comes after the op set's own launch, which a
        # CPU tensor does not reach
        with pytest.raises(ValueError):
            model.attention_core(0, qkv, torch.zeros(3, dtype=torch.int32), None, _batch())
        assert "append" not in log and "appended" not in log
        return
    model.attention_core(0, qkv, None, None, _batch())
    if kind == "plain":
        assert log == ["layer_kv", "append", "appended"]
    else:
        assert "append" not in log and log[-1] == "forward" and "rope" in log


class _NoLaunch:
    def __getattr__(self, name):
        return lambda *args: 0


@pytest.mark.parametrize("how", ["subclass", "attribute"])
@pytest.mark.parametrize("name,rows,k,silu", [("fused_add_rmsnorm", 8, 2560, False),
                                              ("linear", 8, 2560, True),
                                              ("silu_and_mul", 24, 1280, True)])
def test_own_parts_of_the_norm_and_projection_are_called(how, name, rows, k, silu, monkeypatch):
    """add_rmsnorm_linear outside the folded launch goes through the op set's own
    residual-add norm, projection and activation."""
    monkeypatch.setattr(_lib, "lib", lambda: _NoLaunch())
    monkeypatch.setattr(_lib, "raw_stream", lambda t: 0)
    empty, like = torch.empty, torch.empty_like
    monkeypatch.setattr(torch, "empty", lambda *a, **k: empty(*a, **k).as_subclass(_GpuTensor))
    monkeypatch.setattr(torch, "empty_like", lambda x: like(x).as_subclass(_GpuTensor))
    log = []

    def own(*args):
        log.append(name)
        return getattr(HipOps, name)(*args)

    if how == "subclass":
        ops = type("Own", (HipOps,), {name: staticmethod(own)})()
    else:
        ops = _with(HipOps(), **{name: own})
    t = lambda *shape: torch.zeros(shape, dtype=BF).as_subclass(_GpuTensor)
    ops.add_rmsnorm_linear(t(rows, k), t(rows, k), t(k), 1e-6, t(64, k), silu=silu)
    assert log == [name]
