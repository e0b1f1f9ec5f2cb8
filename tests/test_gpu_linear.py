"""GPU parity of ckv_linear (ops.linear) against fp64 torch, and of the calls that ops.linear leaves
to torch.

Tolerance per element: one bf16 rounding of the result (2^-8 of its size covers the rounding and a
neighbouring tie) plus the fp32 accumulation of K products and the bias, each add rounding to 2^-24
of a partial sum that the sum of absolute products bounds.
"""

import pytest
import torch
import torch.nn.functional as F

from chunkkv_amd import _native, ops
from chunkkv_amd.engine import _apply_linear

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _operands(M, N, K, bias=True, dtype=torch.bfloat16):
    g = torch.Generator(device=DEV).manual_seed(M * 31 + N * 7 + K)
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV).to(dtype)  # noqa: E731
    return rand(1, M, K), rand(N, K), rand(N) if bias else None


def _close(out, x, w, b):
    ref = x.double() @ w.double().t().contiguous()
    size = x.double().abs() @ w.double().abs().t().contiguous()
    if b is not None:
        ref, size = ref + b.double(), size + b.double().abs()
    bound = ref.abs() * 2.0**-8 + size * (x.shape[-1] + 1) * 2.0**-24 + 1e-30
    assert bool(((out.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("M,N,K,bias", [
    (2, 8, 64, True),        # one step, one column group, two rows
    (63, 72, 128, False),    # ragged tile both ways
    (64, 64, 256, True),     # exactly one tile and one group of steps
    (65, 136, 320, True),    # one row past a tile, a group and one step
    (251, 1152, 896, True),  # q|k|v of the 0.5B shape
    (251, 896, 4864, False), # down: K split in four
    (3, 896, 4864, True),    # K split in eight, bias added by the sum
    (1103, 896, 896, False),
    (17, 3584, 3584, True),
])
def test_linear_matches_fp64(M, N, K, bias):
    x, w, b = _operands(M, N, K, bias)
    assert _native.lib().ckv_linear_workspace_bytes(M, N, K) >= 0
    out = ops.linear(x, w, b)
    assert out.shape == (1, M, N) and out.dtype == torch.bfloat16
    _close(out, x, w, b)
    assert torch.equal(out[0], ops.linear(x[0], w, b))


def test_linear_unsplit_without_workspace():
    x, w, b = _operands(20, 896, 4864)
    out = torch.empty(20, 896, dtype=torch.bfloat16, device=DEV)
    st = torch.cuda.current_stream().cuda_stream
    assert _native.lib().ckv_linear_workspace_bytes(20, 896, 4864) > 0
    assert _native.lib().ckv_linear(out.data_ptr(), x.data_ptr(), 4864, w.data_ptr(), b.data_ptr(), 20, 896, 4864,
                                    _native.DTYPE_BF16, None, 0, st) == _native.CKV_OK
    _close(out[None], x, w, b)


@pytest.mark.parametrize("M,N,K,dtype,change", [
    (1, 896, 896, torch.bfloat16, None),        # one row: the library's
    (1103, 9728, 896, torch.bfloat16, None),    # large: the library's
    (10, 64, 96, torch.bfloat16, None),         # K not in whole steps
    (10, 60, 64, torch.bfloat16, None),         # N not in eights
    (10, 64, 64, torch.float32, None),
    (10, 64, 64, torch.bfloat16, lambda x, w: (x[:, ::2], w)),            # rows apart
    (10, 64, 64, torch.bfloat16, lambda x, w: (x, w.t())),                # transposed weight
    (10, 64, 65, torch.bfloat16, lambda x, w: (x[..., 1:], w[:, 1:])),    # unaligned rows
])
def test_linear_leaves_the_rest_to_torch(M, N, K, dtype, change):
    x, w, b = _operands(M, N, K, dtype=dtype)
    if change is not None:
        x, w = change(x, w)
    assert torch.equal(ops.linear(x, w, b), F.linear(x, w, b))


def test_linear_keeps_gradients_and_wrapped_modules():
    x, w, b = _operands(10, 64, 64)
    w.requires_grad_(True)
    ops.linear(x, w, b).float().sum().backward()
    assert w.grad is not None
    m = torch.nn.Linear(64, 64, device=DEV, dtype=torch.bfloat16)
    with torch.inference_mode():
        assert torch.equal(_apply_linear(m, x), ops.linear(x, m.weight, m.bias))
        seen = []
        m.register_forward_hook(lambda *a: seen.append(1))
        _apply_linear(m, x)
        assert seen == [1]


def test_linear_under_transforms_equals_torch():
    """Autocast of another type, vmap, forward-mode tangents: as torch's own call, at a size that
    ckv_linear takes without them."""
    import torch.autograd.forward_ad as fw

    x, w, b = _operands(10, 64, 64)
    with torch.autocast("cuda", torch.float16):
        y = ops.linear(x, w, b)
        assert y.dtype == torch.float16 and torch.equal(y, F.linear(x, w, b))
    with torch.autocast("cuda", torch.bfloat16):
        assert torch.equal(ops.linear(x.float(), w, b), F.linear(x.float(), w, b))
    xs = torch.stack([x[0], -x[0]])
    assert torch.equal(torch.func.vmap(lambda a: ops.linear(a, w, b))(xs), torch.func.vmap(lambda a: F.linear(a, w, b))(xs))
    with fw.dual_level():
        d = fw.make_dual(x, x.flip(1))
        got, want = (fw.unpack_dual(f(d, w, b)) for f in (ops.linear, F.linear))
        assert torch.equal(got.primal, want.primal) and torch.equal(got.tangent, want.tangent)
