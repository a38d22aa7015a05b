"""GPU parity of the wave-split kernel (csrc/attn_fwd_wavesplit.hpp): few rows per KV head and
small grids at the default tiles. At the edges of its row tiles (32 and 64 rows), of its key tiles
(32, 64, 128 keys by head_dim) and of the key groups' turns, against the oracle with the reference's
rule, and against the general kernel on the same inputs (127 rows a program keep a call off the
wave-split kernel).
"""

import pytest
import torch

from attn_check import check_against_oracle, make_qkv
from oracle import reference as ref

pytestmark = pytest.mark.gpu

LSE_ATOL = 1e-4  # tests/test_gpu_splitkv.py


def _attention():
    from fa2.kernel import attention
    return attention


def _check(q, k, v, causal):
    attention = _attention()
    out, lse = attention(q, k, v, causal=causal, return_lse=True)
    assert torch.equal(out, attention(q, k, v, causal=causal))
    check_against_oracle(q, k, v, causal, ours=out)
    want = ref.naive_lse(q.double(), k.double(), None, causal=causal)
    assert (lse.double() - want).abs().max().item() <= LSE_ATOL
    general = attention(q, k, v, causal=causal, block_m=127, pack_gqa=False, num_splits=1)
    check_against_general(out, general)


def check_against_general(out, general):
    """The 2-norm of the difference, over all outputs and per query head, against the output's own. Each
    kernel rounds every weight P and the output to the input type, relative errors of u / sqrt(3) = 0.58 u
    at most in the mean square (u = 2^-8 in bf16, 2^-11 in fp16); independent values make an output and the
    error of its weights sums over the same weights, so the error is that share of the output whatever
    the key count. Two roundings in two kernels: 1.2 u, within 2 u over all outputs, and within 4 u of a
    head, which may have as few as 16. A key group left out would leave half of the output or more."""
    u = 2.0 ** (-8 if out.dtype == torch.bfloat16 else -11)
    diff, ref_ = (out.double() - general.double()), general.double()
    assert diff.norm().item() <= 2 * u * ref_.norm().item()
    assert (diff.flatten(2).norm(dim=2) <= 4 * u * ref_.flatten(2).norm(dim=2)).all()


# rows per KV head (n_q * group) below, at and past 32 and 64; key counts at the edges of a tile and
# of a round of the four key groups (128 / 256 / 512 keys), one and several splits
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [16, 32, 64, 128])
@pytest.mark.parametrize("h_q,h_kv,n_q,n_kv", [
    (8, 2, 1, 129), (8, 2, 8, 255), (8, 2, 8, 512), (28, 4, 1, 1537), (20, 4, 7, 300), (6, 2, 11, 193),
    (8, 8, 32, 321), (4, 4, 33, 640), (8, 2, 16, 1000), (5, 1, 13, 4100), (2, 2, 64, 9000),
    (8, 1, 1, 3000), (4, 4, 333, 1500), (8, 2, 65, 2048)])
def test_full(dtype, D, h_q, h_kv, n_q, n_kv):
    _check(*make_qkv(2, h_q, h_kv, n_q, n_kv, D, dtype), causal=False)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [16, 32, 64, 128])
@pytest.mark.parametrize("B,h_q,h_kv,n", [
    (1, 4, 4, 129), (2, 8, 2, 193), (1, 4, 1, 256), (3, 5, 1, 383), (1, 28, 4, 400), (1, 8, 2, 1000),
    (2, 16, 16, 520), (1, 32, 8, 1030)])
def test_causal(dtype, D, B, h_q, h_kv, n):
    _check(*make_qkv(B, h_q, h_kv, n, n, D, dtype), causal=True)


# one shape per branch of the rule where 32-row workgroups outnumber the CUs (33 to 64 rows, then fewer)
# where the group does not divide 128 (small grid, long keys with splits, large grid), and two to three
# 64-row workgroups per CU (which head_dim 16 and 32 take)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [16, 32, 64, 128])
@pytest.mark.parametrize("B,h_q,h_kv,n_q,n_kv", [
    (17, 8, 8, 40, 300), (33, 16, 8, 20, 1100), (33, 28, 4, 7, 700), (33, 8, 8, 1, 1601), (34, 8, 8, 30, 230),
    (1, 28, 4, 10, 4300), (8, 28, 4, 40, 6200), (20, 28, 4, 30, 4200), (4, 8, 8, 1201, 520), (1, 20, 4, 2000, 4100)])
def test_full_past_one_workgroup_per_cu(dtype, D, B, h_q, h_kv, n_q, n_kv):
    _check(*make_qkv(B, h_q, h_kv, n_q, n_kv, D, dtype), causal=False)


def test_many_units_and_strided_storage():
    """More units than CUs, an odd unit count, and [B, N, H, D] storage."""
    attention = _attention()
    for causal, shape in ((False, (37, 16, 8, 2, 500, 64)), (False, (3, 12, 12, 512, 512, 64)),
                          (True, (3, 12, 12, 512, 512, 64)), (False, (1, 16, 16, 512, 512, 128))):
        q, k, v = make_qkv(*shape, torch.bfloat16)
        want = attention(q, k, v, causal=causal)
        check_against_oracle(q, k, v, causal, ours=want)
        qs, ks, vs = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k, v))
        assert torch.equal(attention(qs, ks, vs, causal=causal), want)


@pytest.mark.parametrize("causal", [True, False])
def test_scores_that_rise_and_extreme_keys(causal):
    """Keys that grow along the sequence move every group's reference on every tile; a key row of
    +/-inf or NaN makes the rows that see it NaN, as the general kernel does, and no other."""
    attention = _attention()
    q, k, v = make_qkv(1, 8, 2, 600, 600, 64, torch.float16)
    ramp = torch.linspace(0.0, 6.0, 600, device=q.device)[:, None].half()
    check_against_oracle(q, k + ramp * q[:, :2].mean(dim=2, keepdim=True), v, causal)
    for bad in (float("inf"), float("nan")):
        kb = k.clone()
        kb[:, 1, 450] = bad
        out = attention(q, kb, v, causal=causal)
        general = attention(q, kb, v, causal=causal, block_m=127, pack_gqa=False, num_splits=1)
        assert torch.equal(out[:, :4].isnan(), general[:, :4].isnan())
        assert not out[:, :4].isnan().any()
        if causal:
            assert not out[:, 4:, :450].isnan().any()
        if bad != bad:
            assert out[:, 4:, 450 if causal else 0:].isnan().all()


# a 32-row and a 64-row launch of each masking, several splits, and both key-tile widths
@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("causal,shape", [(True, (1, 8, 2, 600, 600)), (True, (2, 16, 16, 520, 520)),
                                          (False, (1, 8, 2, 150, 600)), (False, (17, 8, 8, 40, 600)),
                                          (False, (1, 8, 2, 13, 4100))])
@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
def test_non_finite_keys_and_values_as_the_general_kernel(D, causal, shape, bad):
    """One element of one key or value row: every head's NaN and infinite outputs and its finite ones are
    the general kernel's. A masked key of a tile that is read multiplies its value by zero, which is NaN
    for such a value in either kernel; the kernels' last tiles are not of one width, so there the rows
    before the value are NaN in no more places than the general kernel's."""
    from ablation import launch_plan
    from fa2 import _lib

    B, h_q, h_kv, n_q, n_kv = shape
    splits = 1 if causal else _lib.num_splits(*shape, D, causal, 128, 0, 256)
    plan = launch_plan(*shape, D, 0, causal, num_splits=splits,
                       workspace_bytes=_lib.workspace_bytes(B, h_q, n_q, D, splits))
    assert plan["kernel"] == "fa2::attn_wave_split_kernel"
    attention = _attention()
    at = 450
    for dtype in (torch.float16, torch.bfloat16):
        q, k, v = make_qkv(*shape, D, dtype)
        q = torch.where(q == 0, torch.ones_like(q), q)  # inf * 0 would be NaN for the key's sign test
        kb = k.clone()
        kb[:, 1, at, 0] = bad
        out = attention(q, kb, v, causal=causal)
        general = attention(q, kb, v, causal=causal, block_m=127, pack_gqa=False, num_splits=1)
        assert torch.equal(out.isnan(), general.isnan())
        keep = ~general.isnan()
        check_against_general(out.masked_fill(~keep, 0), general.masked_fill(~keep, 0))
        # a score of +inf or NaN makes its row NaN, one of -inf leaves the row's other keys
        sees = torch.zeros_like(out, dtype=torch.bool)
        group = h_q // h_kv
        sees[:, group:2 * group, at if causal else 0:] = True
        hit = sees if bad != bad else sees & (q[..., :1] * bad > 0)
        assert torch.equal(out.isnan(), hit)

        vb = v.clone()
        vb[:, 1, at, 3] = bad
        out = attention(q, k, vb, causal=causal)
        general = attention(q, k, vb, causal=causal, block_m=127, pack_gqa=False, num_splits=1)
        assert not (out.isnan() & ~general.isnan()).any()
        keep = general.isfinite()
        assert torch.equal(out.nan_to_num(0, 0, 0)[keep], out[keep])
        check_against_general(out.masked_fill(~keep, 0), general.masked_fill(~keep, 0))
        column = out[:, group:2 * group, at if causal else 0:, 3]  # the rows that weigh the value
        assert (column.isnan() if bad != bad else column == bad).all()
        assert torch.equal(column.isnan(), general[:, group:2 * group, at if causal else 0:, 3].isnan())
