"""attention()'s native common call (csrc/fa2_torch.cpp) against its Python path: the same bits,
strides and dtypes over every form the native call accepts, and None (so that Python makes the
call) for every form it leaves alone.
"""

import pytest
import torch

from attn_check import make_qkv

pytestmark = pytest.mark.gpu


@pytest.fixture
def both(monkeypatch):
    """(native call, attention() without it)."""
    from fa2 import _lib
    from fa2.kernel import attention

    assert _lib.fast_call is not None, "fa2/_torch_call.so is not built for this torch"
    native = _lib.fast_call

    def python(*a, **kw):
        monkeypatch.setattr(_lib, "fast_call", None)
        try:
            return attention(*a, **kw)
        finally:
            monkeypatch.setattr(_lib, "fast_call", native)

    return native, python


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("lse", [False, True])
@pytest.mark.parametrize("shape,causal", [
    ((1, 4, 4, 256, 256, 64), True), ((2, 28, 4, 1, 3000, 64), False), ((1, 32, 8, 16, 9000, 128), False),
    ((2, 8, 1, 1, 1, 16), True), ((3, 6, 2, 77, 401, 32), False), ((1, 32, 8, 2048, 2048, 128), True),
    ((4, 16, 16, 1024, 1024, 64), False), ((1, 32, 8, 4096, 4096, 128), True)])
def test_same_bits_as_python(both, dtype, lse, shape, causal):
    native, python = both
    q, k, v = make_qkv(*shape, dtype)
    storage = torch.empty(shape[0], 2, shape[3], shape[1], shape[5], dtype=dtype, device="cuda")
    forms = [(q, k, v),
             tuple(t.transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k, v)),
             (storage[:, 1].transpose(1, 2).copy_(q), k, v)]  # half of a larger buffer: out is dense
    for form in forms:
        for scale in (None, 0.2):
            got = native(*form, causal, scale, lse)
            want = python(*form, causal=causal, sm_scale=scale, return_lse=lse)
            got, want = (got, want) if lse else ((got,), (want,))
            for a, b in zip(got, want):
                assert torch.equal(a, b) and a.dtype == b.dtype and a.stride() == b.stride()


def test_same_bits_where_the_key_norm_table_keeps_the_split_count(both):
    """A group of 56 does not pack into 128 rows: without the table the wave-split kernel would take
    two splits; with it (bf16, long keys) the general kernel takes all four asked for."""
    native, python = both
    q, k, v = make_qkv(1, 56, 1, 150, 32768, 128, torch.bfloat16)
    assert torch.equal(native(q, k, v, False, None, False), python(q, k, v, causal=False))


def test_side_stream_and_grad(both):
    native, python = both
    q, k, v = make_qkv(1, 8, 2, 500, 500, 64, torch.bfloat16)
    want = python(q, k, v, causal=True)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        got = native(q.requires_grad_(), k, v, True, None, False)
    torch.cuda.current_stream().wait_stream(s)
    assert torch.equal(got, want) and not got.requires_grad


def test_left_to_python(both):
    native, _ = both
    q, k, v = make_qkv(1, 4, 2, 64, 64, 64, torch.float16)

    class Sub(torch.Tensor):
        pass

    odd = torch.empty(1, 4, 64, 68, dtype=q.dtype, device="cuda")[..., :64]     # rows of 136 bytes
    off = torch.empty(1 * 4 * 64 * 64 + 1, dtype=q.dtype, device="cuda")[1:].view(1, 4, 64, 64)
    wide = torch.empty((1 << 22) + 72, dtype=q.dtype, device="cuda").as_strided(
        (1, 2, 2, 64), (0, 0, (1 << 22) + 8, 1))
    for bad in [(q.cpu(), k.cpu(), v.cpu(), True, None, False), (q.float(), k.float(), v.float(), True, None, False),
                (q, k, v.bfloat16(), True, None, False), (q[0], k[0], v[0], True, None, False),
                (q[:, :3], k, v, True, None, False), (q[:, :, :5], k, v, True, None, False),
                (q[:, :, :0], k[:, :, :0], v[:, :, :0], True, None, False), (q, k, v, True, -1.0, False),
                (q, k, v, True, 1, False), (q.as_subclass(Sub), k, v, True, None, False),
                (odd, k, v, True, None, False), (off, k, v, True, None, False),
                (q[:, :, :2], wide, wide, False, None, False), (q, k, None, True, None, False)]:
        assert native(*bad) is None
    with torch.overrides.TorchFunctionMode():
        assert native(q, k, v, True, None, False) is None
