"""The native per-layer calls (chunkkv_amd/csrc/torch_ops.cpp) on operands that cannot be launched,
with no GPU: each ends in a Python exception, and the process goes on.

The operands are fake tensors of a HIP device (shape, type and device, no memory), plain and under
torch.func.vmap: the address or stream lookup inside the call fails after all its checks. A call that
mishandles this ends the whole process, so every one runs in a child.
"""

import os
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]

PRELUDE = """
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from chunkkv_amd import ops
BF, I64, I32, U8 = torch.bfloat16, torch.int64, torch.int32, torch.uint8
def t(*shape, dtype=BF):
    return torch.empty(shape, dtype=dtype, device="cuda")
def slab():
    return t(3, 1, 2, 64, 64)
def batched(fn, x):
    return torch.func.vmap(fn)(torch.stack([x, x]))
def repair(k):
    return ops.layer1_repair_gather(slab(), slab(), t(6, dtype=I64), 1, (2, 3), t(6, dtype=I32), 1, 64, k, t(1, 2, 64, 64),
                                    t(64, dtype=U8), t(64, dtype=I32), t(4, dtype=I32), None, 1e6, t(1 << 22, dtype=I32))
CALLS = {
    "attention_active": lambda wrap: wrap(lambda q: ops.attention_active(q, t(1, 2, 64, 64), t(1, 2, 64, 64), t(8, dtype=I64)),
                                          t(1, 4, 8, 64)),
    "rope_qkv": lambda wrap: wrap(lambda q: ops.rope_qkv(q, t(1, 8, 128), None, t(8, dtype=I64), 4, 2, 64, 1e6), t(1, 8, 256)),
    "add_rmsnorm": lambda wrap: wrap(lambda h: ops.add_rmsnorm(h, None, t(64), 1e-6), t(4, 64)),
    "silu_mul": lambda wrap: wrap(lambda g: ops.silu_mul(g, t(4, 64)), t(4, 64)),
    "linear": lambda wrap: wrap(lambda x: ops.linear(x, t(64, 64)), t(4, 64)),
    "layer1_repair_gather": lambda wrap: wrap(repair, t(1, 2, 64, 64)),
    "extract_chunks": lambda wrap: wrap(lambda k: ops.extract_chunks(k, slab(), [(0, 8)]), slab()),
    "extract_chunks_many": lambda wrap: wrap(lambda k: ops.extract_chunks(k, slab(), [(0, 8)] * 65), slab()),
}
"""


def _child(body: str) -> str:
    env = dict(os.environ, HIP_VISIBLE_DEVICES="-1")  # no device, also where there is one
    r = subprocess.run([sys.executable, "-c", PRELUDE + body], cwd=ROOT, env=env, capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0, (r.returncode, r.stdout[-2000:], r.stderr[-2000:])
    return r.stdout


@pytest.mark.parametrize("wrap", ["lambda fn, x: fn(x)", "batched"], ids=["plain", "vmap"])
def test_failing_lookups_raise(wrap):
    out = _child(f"""
with FakeTensorMode():
    for name, call in CALLS.items():
        try:
            call({wrap})
            print(name, "returned", flush=True)
        except Exception as e:
            print(name, "raised", type(e).__name__, str(e).splitlines()[0][:100], flush=True)
""")
    lines = [line.split() for line in out.splitlines()]
    want = ["attention_active", "rope_qkv", "add_rmsnorm", "silu_mul", "linear", "layer1_repair_gather",
            "extract_chunks", "extract_chunks_many"]
    assert [line[0] for line in lines] == want
    # torch computes a product of fake tensors as a fake tensor: linear may return one
    assert all(line[1] == "raised" or line[0] == "linear" for line in lines), out


def test_linear_leaves_transforms_modes_and_subclasses_to_torch():
    """Products that ckv_linear would take by type and shape, on fake tensors: whatever sits between a
    call and the device takes part as in torch.nn.functional.linear."""
    out = _child("""
import torch.autograd.forward_ad as fw
from torch.overrides import TorchFunctionMode
seen = []
class Functions(TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        seen.append(func.__name__)
        return func(*args, **(kwargs or {}))
class Wrapped(torch.Tensor):
    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        seen.append(func.__name__)
        return "wrapped"
with FakeTensorMode():
    x, w = t(10, 64), t(64, 64)
    y = ops.linear(x, w)
    assert type(y).__name__ == "FakeTensor" and y.shape == (10, 64) and y.dtype == BF
    y = batched(lambda a: ops.linear(a, w), x)
    assert y.shape == (2, 10, 64)
    with fw.dual_level():
        for args in ((fw.make_dual(x, t(10, 64)), w), (x, fw.make_dual(w, t(64, 64))), (x, w, fw.make_dual(t(64), t(64)))):
            assert fw.unpack_dual(ops.linear(*args)).tangent is not None
    with Functions():
        ops.linear(x, w)
    assert seen == ["linear"], seen
assert ops.linear(torch.zeros(4, 64).as_subclass(Wrapped), torch.zeros(64, 64)) == "wrapped"
print("ok")
""")
    assert out.strip() == "ok"


def test_apply_linear_calls_what_is_not_a_plain_linear(monkeypatch):
    """HipEngine's shortcut past nn.Linear.__call__ is taken for nothing that changes what the call
    does."""
    import torch

    from chunkkv_amd import engine, ops

    monkeypatch.setattr(ops, "linear", lambda *a: "shortcut")
    x, made = torch.zeros(2, 8), lambda: torch.nn.Linear(8, 8)
    assert engine._apply_linear(made(), x) == "shortcut"

    hooked, compiled, replaced, moved = made(), made(), made(), made()
    hooked.register_forward_hook(lambda *a: "hook")
    compiled._compiled_call_impl = lambda *a: "compiled"
    replaced.forward = lambda *a: "forward"
    bias = moved._parameters.pop("bias").detach()
    moved.bias = bias + 1.0
    assert engine._apply_linear(hooked, x) == "hook"
    assert engine._apply_linear(compiled, x) == "compiled"
    assert engine._apply_linear(replaced, x) == "forward"
    assert torch.equal(engine._apply_linear(moved, x), (bias + 1.0).expand(2, 8))
    monkeypatch.setattr(torch.nn.Linear, "forward", lambda *a: "class")
    assert engine._apply_linear(made(), x) == "class"
