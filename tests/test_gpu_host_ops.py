"""The native launch path (csrc/host_ops.cpp) against the general one.

Every call below runs twice: with the native module, and with one that
handles nothing, so that the Python checks and the ctypes launch serve it.
Both must give the same bits, shapes and strides, or raise the same error.
"""

import types

import pytest
import torch

from my_vllm_amd import _native, ops
from my_vllm_amd.attention_backend import MI355XAttentionBackend
from workloads import make_paged_batch

pytestmark = pytest.mark.gpu

NAMES = ("silu_and_mul", "rms_norm", "fused_add_rms_norm", "qk_norm_rope_store", "paged_decode", "paged_prefill",
         "paged_mixed", "forward_inputs_ok")


def outcome(call):
    try:
        out = call()
    except Exception as error:  # the two paths must agree on the error too
        return type(error), str(error)
    out = out if isinstance(out, tuple) else (out,)
    return [(t.shape, t.stride(), t.dtype, t.clone()) for t in out if t is not None]


def both(monkeypatch, make):
    """``make()`` builds a call on fresh inputs; returns whether the native
    module took it."""
    taken = []
    real = _native.host_ops()

    def spy(name):
        def f(*a):
            r = getattr(real, name)(*a)
            taken.append((name, r is not None))
            return r
        return f

    results = []
    for module in (types.SimpleNamespace(**{n: spy(n) for n in NAMES}),
                   types.SimpleNamespace(**{n: lambda *a: None for n in NAMES})):
        with monkeypatch.context() as m:
            m.setattr(_native, "_host", module)
            results.append(outcome(make()))
    fast, general = results
    if isinstance(general, tuple):
        assert fast == general
    else:
        assert len(fast) == len(general)
        for a, b in zip(fast, general):
            assert a[:3] == b[:3] and torch.equal(a[3], b[3])
    return any(ok for name, ok in taken if name != "forward_inputs_ok")


def rand(gpu, *shape, dtype=torch.bfloat16, seed=3):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(dtype).to(gpu)


class Wrapped(torch.Tensor):
    pass


def layer_forms(gpu):
    x = lambda *s, **k: rand(gpu, *s, **k)  # noqa: E731
    bf, fp, f32 = torch.bfloat16, torch.float16, torch.float32
    w = x(512, seed=5)
    return {
        # name: (call factory, whether the native module must take it)
        "silu": (lambda: (lambda: ops.silu_and_mul(x(3, 7, 64))), True),
        "silu 1-D fp16": (lambda: (lambda: ops.silu_and_mul(x(64, dtype=fp))), True),
        "silu odd": (lambda: (lambda: ops.silu_and_mul(x(3, 7))), False),
        "silu empty": (lambda: (lambda: ops.silu_and_mul(x(0, 8))), False),
        "silu strided": (lambda: (lambda: ops.silu_and_mul(x(8, 128)[:, :64])), False),
        "silu fp32": (lambda: (lambda: ops.silu_and_mul(x(8, 64, dtype=f32))), False),
        "silu host": (lambda: (lambda: ops.silu_and_mul(x(8, 64).cpu())), False),
        "silu subclass": (lambda: (lambda: ops.silu_and_mul(x(8, 64).as_subclass(Wrapped)).as_subclass(torch.Tensor)),
                          False),
        "rms 2-D": (lambda: (lambda: ops.rms_norm(x(5, 512), w, 1e-6)), True),
        "rms one strided row": (lambda: (lambda: ops.rms_norm(x(1, 1024)[:, :512], w, 1e-6)), True),
        "rms strided rows, fp32 weight": (lambda: (lambda: ops.rms_norm(x(5, 1024)[:, 512:], w.float(), 1e-6)), True),
        "rms heads": (lambda: (lambda: ops.rms_norm(x(6, 9, 512)[:, 2:5], w, 1e-6)), True),
        "rms every other head": (lambda: (lambda: ops.rms_norm(x(6, 8, 512)[:, ::2], w, 1e-6)), True),
        "rms 1-D": (lambda: (lambda: ops.rms_norm(x(512), w, 1e-6)), False),
        "rms 4-D": (lambda: (lambda: ops.rms_norm(x(2, 3, 4, 512), w, 1e-6)), False),
        "rms empty": (lambda: (lambda: ops.rms_norm(x(0, 512), w, 1e-6)), False),
        "rms weight type": (lambda: (lambda: ops.rms_norm(x(5, 512), w.half(), 1e-6)), False),
        "rms width": (lambda: (lambda: ops.rms_norm(x(5, 256), w, 1e-6)), False),
        "rms inner stride": (lambda: (lambda: ops.rms_norm(x(5, 1024)[:, ::2], w, 1e-6)), False),
        "add": (lambda: (lambda: ops.fused_add_rms_norm(x(5, 512), x(5, 512, seed=4), w, 1e-6)), True),
        "add in place, strided": (lambda: (lambda a=x(5, 1024), b=x(5, 1024, seed=4): ops.fused_add_rms_norm(
            a[:, :512], b[:, 256:768], w, 1e-6, inplace=True)), True),
        "add 3-D": (lambda: (lambda: ops.fused_add_rms_norm(x(2, 5, 512), x(2, 5, 512, seed=4), w, 1e-6)), True),
        "add 3-D strided": (lambda: (lambda: ops.fused_add_rms_norm(x(2, 9, 512)[:, :5], x(2, 5, 512), w, 1e-6)),
                            False),
        "add shapes": (lambda: (lambda: ops.fused_add_rms_norm(x(5, 512), x(4, 512), w, 1e-6)), False),
        "add types": (lambda: (lambda: ops.fused_add_rms_norm(x(5, 512), x(5, 512, dtype=fp), w, 1e-6)), False),
        "add grad": (lambda: (lambda: ops.fused_add_rms_norm(x(5, 512).requires_grad_(), x(5, 512), w, 1e-6)), True),
        "add bf16 eps int": (lambda: (lambda: ops.fused_add_rms_norm(x(5, 512), x(5, 512), w, 1)), False),
        "dtype": (lambda: (lambda: ops.rms_norm(x(5, 512, dtype=bf).double(), w, 1e-6)), False),
    }


LAYER_FORMS = tuple(layer_forms("cpu"))


@pytest.mark.parametrize("name", LAYER_FORMS)
def test_layer_operators(gpu, monkeypatch, name):
    make, native = layer_forms(gpu)[name]
    assert both(monkeypatch, make) is native


@pytest.mark.parametrize("change,native", [
    (None, True), ("int64 slots", True), ("no norm", True), ("fp32 weights", True), ("table 3-D", True),
    ("strided slots", False), ("strided positions", False), ("int32 positions", False), ("v heads", False),
    ("cache type", False), ("one weight", False), ("outputs", True), ("outputs stride", False),
])
def test_prologue(gpu, monkeypatch, change, native):
    def make():
        qkv = rand(gpu, 6, 12, 128)
        q, k, v = qkv.split((8, 2, 2), dim=1)
        a = dict(positions=torch.arange(6, device=gpu), q=q, k=k, cos_sin_cache=rand(gpu, 16, 128, dtype=torch.float32),
                 q_norm_weight=rand(gpu, 128, seed=5), k_norm_weight=rand(gpu, 128, seed=6), eps=1e-6, v=v,
                 k_cache=torch.zeros(2, 16, 2, 128, dtype=q.dtype, device=gpu),
                 v_cache=torch.zeros(2, 16, 2, 128, dtype=q.dtype, device=gpu),
                 slot_mapping=torch.arange(3, 9, dtype=torch.int32, device=gpu))
        if change == "int64 slots":
            a["slot_mapping"] = a["slot_mapping"].long()
        elif change == "strided slots":
            a["slot_mapping"] = torch.arange(12, dtype=torch.int32, device=gpu)[::2]
        elif change == "strided positions":
            a["positions"] = torch.arange(12, device=gpu)[::2]
        elif change == "int32 positions":
            a["positions"] = a["positions"].int()
        elif change == "no norm":
            a["q_norm_weight"] = a["k_norm_weight"] = None
        elif change == "one weight":
            a["k_norm_weight"] = None
        elif change == "fp32 weights":
            a["q_norm_weight"], a["k_norm_weight"] = a["q_norm_weight"].float(), a["k_norm_weight"].float()
        elif change == "table 3-D":
            a["cos_sin_cache"] = a["cos_sin_cache"].unsqueeze(1)
        elif change == "v heads":
            a["v"] = v[:, :, ::2]
        elif change == "cache type":
            a["v_cache"] = a["v_cache"].half()
        elif change == "outputs":
            a["q_out"], a["k_out"], _ = torch.empty_like(qkv).split((8, 2, 2), dim=1)
        elif change == "outputs stride":
            a["q_out"] = torch.empty(6, 8, 128, dtype=q.dtype, device=gpu)

        def call():
            out = ops.qk_norm_rope_store(**a)
            return (*out, a["k_cache"], a["v_cache"])
        return call

    assert both(monkeypatch, make) is native


@pytest.mark.parametrize("prefill", [0, 1, 3])
@pytest.mark.parametrize("change,native", [
    (None, True), ("query stride", True), ("store", True), ("query type", False), ("cache layout", False),
    ("value cache", False), ("int64 slots", True), ("table rows", True),
])
def test_backend_routes(gpu, monkeypatch, prefill, change, native):
    q_lens, kv_lens = [5, 40, 1], [5, 300, 77]
    if prefill == 0:
        q_lens = [1, 1, 1]
    elif prefill == 1:
        q_lens, kv_lens = [40, 1, 1], [300, 5, 77]

    def make():
        batch = make_paged_batch(31, q_lens, kv_lens, prefill, 16, 4)
        c = batch.common
        common = type(c)(**{**c.__dict__, **{n: getattr(c, n).to(gpu) for n in
                                             ("query_start_loc", "seq_lens", "slot_mapping", "block_tables")}})
        backend = MI355XAttentionBackend(16, 4, 128, 16, torch.bfloat16)
        q, k, v, kc, vc = (t.to(gpu) for t in (batch.q, batch.k_new, batch.v_new, batch.k_cache, batch.v_cache))
        slots = common.slot_mapping
        if change == "query stride":
            q = torch.cat((q, q), 1)[:, :16]
        elif change == "query type":
            q = q.half()
        elif change == "cache layout":
            kc, vc = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (kc, vc))
        elif change == "value cache":
            vc = vc[:-1]
        elif change == "int64 slots":
            slots = slots.long()
        elif change == "table rows":
            wide = torch.full((3, 64), -1, dtype=torch.int32, device=gpu)
            wide[:, :common.block_tables.size(1)] = common.block_tables
            common = type(c)(**{**common.__dict__, "block_tables": wide[:, :common.block_tables.size(1)]})
        plan = backend.build_plan(common)

        def call():
            if change in ("store", "int64 slots"):
                return backend.forward_with_kv_store(q, k, v, kc, vc, slots, plan), kc, vc
            return backend.forward(q, k, v, kc, vc, plan)
        return call

    assert both(monkeypatch, make) is native


def test_host_tensors_are_left_to_the_general_path():
    x = torch.zeros(4, 8, dtype=torch.bfloat16)
    host = _native.host_ops()
    assert host.silu_and_mul(x) is None and host.silu_and_mul(None) is None and host.silu_and_mul() is None
    assert host.rms_norm(x, x[0], 1e-6) is None
    assert host.fused_add_rms_norm(x, x, x[0], 1e-6, False) is None
