"""The wide kernel (csrc/attn_fwd_wide.hpp: full attention at head_dim 32 and 64, 256-row programs)
against the general kernel, bit for bit: 127 rows a program keep a call off it, and a row's
arithmetic does not depend on the rows per program. One shape per edge of its range: one round of
programs, a ragged last program and key tile, packing, the log-sum-exp, the key-norm table with rows
that pass and rows that fail, scores that move the reference on every tile. (Accuracy against the
oracle is the general kernel's, tests/test_gpu_parity.py; one shape is checked here as well.)
"""

import pytest
import torch

from attn_check import check_against_oracle, make_qkv

pytestmark = pytest.mark.gpu


def _same_as_general(q, k, v, table=False):
    from fa2 import _lib
    from fa2.kernel import LOG2E, attention

    B, h_q, n, D = q.shape
    h_kv, n_kv = k.shape[1], k.shape[2]
    stream = torch.cuda.current_stream().cuda_stream
    ws = (torch.empty((B * h_kv * ((n_kv + 63) // 64) * 4 + 255) // 256 * 256, dtype=torch.uint8,
                      device=q.device) if table else None)
    res = []
    for bm in (128, 127):
        out = torch.empty_like(q)
        lse = torch.empty(B, h_q, n, device=q.device)
        # the table needs the default 4-wave programs, which 127 rows keep too
        _lib.attn_fwd_ex(q, k, v, out, False, 1, bm, 0, LOG2E / D ** 0.5, lse, 1, ws, stream)
        res.append((out, lse))
    assert torch.equal(res[0][0], res[1][0]) and torch.equal(res[0][1], res[1][1])
    if not table:
        assert torch.equal(attention(q, k, v, causal=False), res[0][0])
    return res[0][0]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("table", [False, True])
@pytest.mark.parametrize("B,h_q,h_kv,n,n_kv", [(8, 16, 16, 1024, 1024), (2, 32, 8, 2047, 1025),
                                               (13, 16, 4, 1000, 1500), (1, 16, 16, 12700, 1090)])
def test_same_bits_as_the_general_kernel(dtype, D, table, B, h_q, h_kv, n, n_kv):
    q, k, v = make_qkv(B, h_q, h_kv, n, n_kv, D, dtype)
    k[:, 0] *= 3.0  # rows of this head fail the table's bound in fp16
    k[:, -1] *= 0.3
    out = _same_as_general(q, k, v, table)
    if B == 8:
        check_against_oracle(q, k, v, False, precision=torch.float32, ours=out)


# shapes that run the wide kernel at both head dims: one round of programs per CU place at 32, ragged
# last programs and key tiles, a grouped and an unpackable head count
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("table", [False, True])
@pytest.mark.parametrize("B,h_q,h_kv,n,n_kv", [(12, 16, 16, 1024, 1024), (3, 32, 8, 2047, 1025),
                                               (15, 16, 4, 1000, 1500), (1, 16, 16, 15700, 1090)])
def test_same_bits_where_the_wide_kernel_runs(dtype, D, table, B, h_q, h_kv, n, n_kv):
    from ablation import launch_plan

    plan = launch_plan(B, h_q, h_kv, n, n_kv, D, 0, False, workspace_bytes=1 << 30 if table else 0)
    assert plan["kernel"] == "fa2::attn_wide_kernel" and plan["key_table"] == table
    q, k, v = make_qkv(B, h_q, h_kv, n, n_kv, D, dtype)
    k[:, 0] *= 3.0  # rows of this head fail the table's bound in fp16
    k[:, -1] *= 0.3
    _same_as_general(q, k, v, table)


@pytest.mark.parametrize("D", [32, 64])
def test_strided_storage(D):
    """[B, N, H, D] storage, and K and V as halves of one buffer: the bits of dense tensors."""
    from ablation import launch_plan
    from fa2.kernel import attention

    B, h_q, h_kv, n, n_kv = 3, 32, 8, 2047, 1025
    plan = launch_plan(B, h_q, h_kv, n, n_kv, D, 1, False)
    assert plan["kernel"] == "fa2::attn_wide_kernel"
    q, k, v = make_qkv(B, h_q, h_kv, n, n_kv, D, torch.bfloat16)
    want = _same_as_general(q, k, v)
    qs, ks, vs = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k, v))
    out = attention(qs, ks, vs, causal=False)
    assert out.stride() == qs.stride() and torch.equal(out, want)
    kv = torch.stack((k.transpose(1, 2), v.transpose(1, 2)), dim=2)  # [B, N, 2, H, D]
    ks, vs = kv[:, :, 0].transpose(1, 2), kv[:, :, 1].transpose(1, 2)
    assert not ks.is_contiguous() and torch.equal(attention(qs, ks, vs, causal=False), want)


@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("table", [False, True])
@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
def test_non_finite_keys_and_values_as_the_general_kernel(D, table, bad):
    """One element of one key and of one value row, bit for bit the general kernel's outputs."""
    from fa2 import _lib
    from fa2.kernel import LOG2E

    B, h_q, h_kv, n, n_kv = 3, 32, 8, 2047, 1025
    stream = torch.cuda.current_stream().cuda_stream
    q, k, v = make_qkv(B, h_q, h_kv, n, n_kv, D, torch.float16)
    ws = torch.empty(1 << 20, dtype=torch.uint8, device=q.device) if table else None
    for t in (k, v):
        saved = t[:, 1, 450, 3].clone()
        t[:, 1, 450, 3] = bad
        res = []
        for bm in (128, 127):
            out = torch.empty_like(q)
            _lib.attn_fwd_ex(q, k, v, out, False, 1, bm, 0, LOG2E / D ** 0.5, None, 1, ws, stream)
            res.append(out)
        assert torch.equal(res[0].isnan(), res[1].isnan()) and res[0].isnan().any() == (t is k or bad != bad)
        assert torch.equal(res[0].nan_to_num(0.0), res[1].nan_to_num(0.0))
        t[:, 1, 450, 3] = saved


def test_reference_moves_on_every_tile_and_packed_rows():
    from fa2.kernel import attention

    q, k, v = make_qkv(8, 16, 8, 1024, 1024, 64, torch.bfloat16)
    k = k + torch.linspace(0.0, 40.0, 1024, device=k.device)[:, None].bfloat16() * q[:, ::2].mean(
        dim=2, keepdim=True)
    out = _same_as_general(q, k, v)
    assert torch.equal(out, attention(q, k, v, causal=False, pack_gqa=True))
