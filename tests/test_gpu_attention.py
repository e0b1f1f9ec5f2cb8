"""GPU parity of the position-masked GQA attention kernel (ckv_attention_active) against the
fp64 oracle and against torch's own SDPA call with the reference's boolean mask.

Tolerance: bf16 inputs and output; the softmax weights are rounded to bf16 before the second
product (relative error 2^-9 per weight), so with N(0, 1) inputs the output is within
1e-2 absolute of the exact fp64 value (the same bound holds for torch's fused bf16 SDPA).
"""

import numpy as np
import pytest
import torch
import torch.nn.functional as F

from chunkkv_amd import _native, ops
from oracle import oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda"
ATOL = 1e-2


def _case(seed, Hq, Hkv, D, N, n, sorted_=True, with_ends=True):
    rng = np.random.default_rng(seed)
    q = O.f32_to_bf16_bits(rng.standard_normal((Hq, n, D)).astype(np.float32))
    K = O.f32_to_bf16_bits(rng.standard_normal((Hkv, N, D)).astype(np.float32))
    V = O.f32_to_bf16_bits(rng.standard_normal((Hkv, N, D)).astype(np.float32))
    pos = rng.choice(N, n, replace=False) if n <= N else rng.integers(0, N, n)
    if with_ends and n >= 2:
        pos[0], pos[-1] = 0, N - 1
    pos = np.sort(pos) if sorted_ else pos
    return q, K, V, pos.astype(np.int64)


def _run(q, K, V, pos):
    err = torch.zeros(1, dtype=torch.int32, device=DEV)
    out = ops.attention_active(O.from_numpy(q, DEV)[None], O.from_numpy(K, DEV)[None], O.from_numpy(V, DEV)[None],
                               torch.from_numpy(pos).to(DEV), err=err)
    torch.cuda.synchronize()
    return out, int(err.item())


@pytest.mark.parametrize(
    "Hq,Hkv,D,N,n",
    [
        (28, 4, 128, 8256, 2976),  # Qwen2.5-7B layer >= 2 of the 8k request
        (28, 4, 128, 1000, 1000),  # every position active (plain causal)
        (14, 2, 64, 1056, 200),  # Qwen2.5-0.5B heads
        (8, 1, 128, 77, 1),  # one query, partial tile
        (4, 4, 64, 130, 129),  # no grouping, ragged tiles
        (7, 7, 128, 64, 3),  # exactly one tile
    ],
)
def test_attention_matches_oracle(Hq, Hkv, D, N, n):
    q, K, V, pos = _case(Hq * 1000 + N, Hq, Hkv, D, N, n)
    out, e = _run(q, K, V, pos)
    assert e == 0
    got = out[0].float().cpu().numpy()
    sub = slice(None) if n <= 600 else np.sort(np.random.default_rng(0).choice(n, 600, replace=False))
    want = O.attention_active(q[:, sub], K, V, pos[sub])
    np.testing.assert_allclose(got[sub], want, atol=ATOL, rtol=0)


def test_attention_unsorted_positions_and_matches_torch_sdpa():
    """Positions in any order give the same rows; the result agrees with torch's SDPA on the
    reference's boolean mask with the KV heads expanded."""
    Hq, Hkv, D, N, n = 28, 4, 128, 700, 300
    q, K, V, pos = _case(5, Hq, Hkv, D, N, n, sorted_=False)
    out, e = _run(q, K, V, pos)
    assert e == 0
    perm = np.argsort(pos)
    out2, _ = _run(np.ascontiguousarray(q[:, perm]), K, V, pos[perm])
    assert torch.equal(out[0][torch.from_numpy(perm).to(DEV)], out2[0])
    qt, Kt, Vt = (O.from_numpy(a, DEV)[None] for a in (q, K, V))
    p = torch.from_numpy(pos).to(DEV)
    mask = p[:, None] >= torch.arange(N, device=DEV)[None, :]
    ref = F.scaled_dot_product_attention(qt, Kt.repeat_interleave(7, 1), Vt.repeat_interleave(7, 1), attn_mask=mask)
    torch.testing.assert_close(out[0].float(), ref[0].transpose(0, 1).float(), atol=2 * ATOL, rtol=0)


def test_attention_flags_out_of_range_position():
    q, K, V, pos = _case(9, 4, 2, 64, 50, 10)
    pos[3] = 50
    _, e = _run(q, K, V, pos)
    assert e == _native.DEVICE_ERR_RANGE


def test_attention_strided_query_view():
    """q as the transposed view of a token-major projection output (rows contiguous)."""
    Hq, Hkv, D, N, n = 28, 4, 128, 300, 123
    q, K, V, pos = _case(3, Hq, Hkv, D, N, n)
    qt = O.from_numpy(np.ascontiguousarray(q.transpose(1, 0, 2)), DEV)[None].transpose(1, 2)  # (1, Hq, n, D) view
    assert not qt.is_contiguous()
    out = ops.attention_active(qt, O.from_numpy(K, DEV)[None], O.from_numpy(V, DEV)[None], torch.from_numpy(pos).to(DEV))
    ref, _ = _run(q, K, V, pos)
    assert torch.equal(out, ref)


@pytest.mark.parametrize("Hq,Hkv,D,N,n", [
    (28, 4, 128, 8256, 1),  # decode: grouped rows (7 query heads of a KV head per workgroup)
    (28, 4, 128, 5000, 3),  # grouped, 21 rows
    (16, 2, 128, 777, 16),  # grouped, exactly one workgroup of rows (16 x 8), ragged last split
    (14, 2, 64, 3001, 1),   # grouped at head_dim 64 (Qwen2.5-0.5B decode), ragged last tile
    (14, 2, 64, 3000, 40),  # 280 rows: token rows per query head, split
    (8, 8, 64, 3000, 2),    # no grouping (one query head per KV head): token rows, split
])
def test_attention_split_launch_matches_oracle_and_unsplit(Hq, Hkv, D, N, n):
    """Decode-like shapes split the cache range over workgroups and merge: same result as the
    unsplit launch (up to the merge's fp32 rounding) and the oracle. Launches whose queries share
    KV heads and fit one workgroup put the group's query heads in one workgroup's rows."""
    q, K, V, pos = _case(N + n, Hq, Hkv, D, N, n, with_ends=False)
    pos[-1] = N - 1
    assert _native.lib().ckv_attention_workspace_bytes(n, N, Hq, D, None, None) > 0
    args = (O.from_numpy(q, DEV)[None], O.from_numpy(K, DEV)[None], O.from_numpy(V, DEV)[None], torch.from_numpy(pos).to(DEV))
    split = ops.attention_active(*args)
    whole = ops.attention_active(*args, split=False)
    torch.cuda.synchronize()
    torch.testing.assert_close(split.float(), whole.float(), atol=4e-3, rtol=0)
    np.testing.assert_allclose(split[0].float().cpu().numpy(), O.attention_active(q, K, V, pos), atol=ATOL, rtol=0)


@pytest.mark.parametrize("Hq,Hkv,D,N,n", [
    (28, 4, 128, 1, 1),      # one cache row
    (28, 4, 128, 31, 31),    # less than one 32-row chunk
    (12, 3, 64, 33, 17),     # KV heads that do not divide the 8 XCDs; one row past a chunk and past 16 rows
    (28, 4, 128, 320, 320),  # 32 rows a workgroup (more 16-row workgroups than fit at once)
    (14, 2, 64, 200, 200),   # 16 rows a workgroup, last one ragged
    (28, 4, 128, 512, 2),    # one token's worth of rows over 16 chunks: not split
    (28, 4, 128, 513, 2),    # 17 chunks: split, the last split one row long
    (28, 4, 128, 767, 251),  # 24 chunks: eight wavefronts
    (14, 2, 64, 1103, 251),  # eight wavefronts, 16 rows each
    (28, 4, 64, 4100, 150),  # eight wavefronts, 16 rows, 129 chunks
    (28, 4, 128, 1180, 1152),  # 252 128-query workgroups: the last size below the large kernel's range
    (28, 4, 128, 1181, 1153),  # 280: the first inside it
    (16, 16, 64, 2100, 40),  # no grouping, split
    (28, 4, 128, 1408, 1280),  # the large kernel, its last tile three rows past the positions
    (8, 8, 64, 7990, 7950),  # the same at head_dim 64, the last tile also past the cache
])
def test_attention_small_launch_forms(Hq, Hkv, D, N, n):
    """Every form of the small-launch kernel (rows and wavefronts per workgroup, grouped rows, splits)
    at the edges of its range, and the large kernel beyond: against the oracle, unsplit, and with the
    rows past every position uninitialised (NaN), which no query may see. Tolerance as at the top of
    this file."""
    q, K, V, pos = _case(N * 7 + n, Hq, Hkv, D, N, n)
    seen = max(1, N - 3)
    pos = np.minimum(pos, seen - 1)
    K[:, seen:], V[:, seen:] = 0x7FC0, 0x7FC0
    args = [O.from_numpy(a, DEV)[None] for a in (q, K, V)] + [torch.from_numpy(pos).to(DEV)]
    got = ops.attention_active(*args)
    whole = ops.attention_active(*args, split=False)
    sub = np.unique(np.linspace(0, n - 1, min(n, 200)).astype(int))
    want = O.attention_active(q[:, sub], K[:, :seen], V[:, :seen], pos[sub])
    for out in (got, whole):
        np.testing.assert_allclose(out[0].float().cpu().numpy()[sub], want, atol=ATOL, rtol=0)


@pytest.mark.parametrize("Hq,Hkv,D,N,n", [
    (130, 65, 64, 768, 57),   # 114 grouped rows, long cache
    (130, 65, 128, 300, 64),  # 128 grouped rows, short cache
    (146, 73, 128, 1000, 57),
    (160, 80, 64, 40, 50),
])
def test_attention_more_kv_heads_than_a_grouped_launch_fills(Hq, Hkv, D, N, n):
    """More than 64 KV heads, whose grouped launches run the nearest form there is. Tolerance as at
    the top of this file."""
    q, K, V, pos = _case(Hq + n, Hq, Hkv, D, N, n)
    out, e = _run(q, K, V, pos)
    assert e == 0
    np.testing.assert_allclose(out[0].float().cpu().numpy(), O.attention_active(q, K, V, pos), atol=ATOL, rtol=0)


@pytest.mark.parametrize("Hq,Hkv,D,N,n", [
    (28, 4, 128, 5120, 130),  # ten splits of eight tiles, the second query block two rows
    (7, 7, 128, 9001, 700),   # no grouping, the last split and the last tile ragged
    (32, 8, 64, 9000, 251),
    (12, 3, 64, 8300, 333),   # KV heads that do not divide the 8 XCDs
])
def test_attention_large_kernel_in_splits(Hq, Hkv, D, N, n):
    """128-query workgroups over splits of a long cache: against the oracle and unsplit, with a query at
    position 0 (it sees one row of the first split and none of the others) and the rows past every
    position uninitialised (NaN). Tolerance as at the top of this file."""
    q, K, V, pos = _case(N + n, Hq, Hkv, D, N, n)
    seen = N - 3
    pos = np.minimum(pos, seen - 1)
    K[:, seen:], V[:, seen:] = 0x7FC0, 0x7FC0
    args = [O.from_numpy(a, DEV)[None] for a in (q, K, V)] + [torch.from_numpy(pos).to(DEV)]
    sub = np.unique(np.r_[0, 1, np.linspace(0, n - 1, min(n, 120)).astype(int)])
    want = O.attention_active(q[:, sub], K[:, :seen], V[:, :seen], pos[sub])
    for out in (ops.attention_active(*args), ops.attention_active(*args, split=False)):
        np.testing.assert_allclose(out[0].float().cpu().numpy()[sub], want, atol=ATOL, rtol=0)
