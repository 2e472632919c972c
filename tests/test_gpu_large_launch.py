"""Calls whose workgroups hold 2^32 or more work-items in all, which is more than one launch takes: the fp32 forward (16 rows
per workgroup), the column passes (64 or 128 keys) and KeyFormer's row pass (128 rows). Every (batch, head) gets the same
inputs (stride 0), so each result must be that of a call with one head, which the oracle tests cover."""
import pytest
import torch

from deepgengraph_amd import _lib
from deepgengraph_amd import attention as A

pytestmark = pytest.mark.gpu


@pytest.fixture
def shared(gpu):
    """randn(rows, D, ...) of one head, shown as [B, rows, H, D] with stride 0 over batch and head."""
    g = torch.Generator(device=gpu).manual_seed(1)

    def make(B, rows, H, D, dtype):
        return torch.randn(1, rows, 1, D, generator=g, device=gpu).to(dtype).expand(B, rows, H, D)

    yield make
    torch.cuda.empty_cache()


def _one(*tensors):
    return [t[:1, :, :1] for t in tensors]


def test_fp32_forward(gpu, shared):
    B, H, Sq, Sk, D = 64, 64, 65536, 16, 64  # 2^24 workgroups of 256
    q, k, v = shared(B, Sq, H, D, torch.float32), shared(B, Sk, H, D, torch.float32), shared(B, Sk, H, D, torch.float32)
    want = A.attention(*_one(q, k, v), causal=False)
    out = A.attention(q, k, v, causal=False)
    for b in range(B):
        assert torch.equal(out[b], want[0].expand(Sq, H, D)), f"batch {b}"


@pytest.mark.parametrize("epilogue,B,Sq", [(_lib.COL_ANY_GE, 64, 64), (_lib.COL_SUM, 128, 32)])
def test_column_scores(gpu, shared, epilogue, B, Sq):
    H, Sk, D = 64, 131072, 128  # 2^23 workgroups of 512: 64 keys each (COL_ANY_GE), 128 keys (COL_SUM)
    q, k = shared(B, Sq, H, D, torch.float16), shared(B, Sk, H, D, torch.float16)
    kw = dict(epilogue=epilogue, causal=False, ref_rounding=False)
    if epilogue == _lib.COL_ANY_GE:  # probabilities around 1 / Sk, about half of the keys above their thresholds
        g = torch.Generator(device=gpu).manual_seed(2)
        kw["thr"] = torch.rand(Sq, Sk, generator=g, device=gpu) * (40.0 / Sk) + 4.0 / Sk
    _, lse = A.attention(*_one(q, k, k), causal=False, return_lse=True)
    want = A.attention_colscore(*_one(q, k), lse, **kw)
    out = A.attention_colscore(q, k, lse.expand(B, H, Sq).contiguous(), **kw)
    if epilogue == _lib.COL_ANY_GE:
        assert 0.1 < want.float().mean().item() < 0.9
    for b in range(B):
        assert torch.equal(out[b], want[0].expand(H, Sk)), f"batch {b}"


def test_keyformer_rows(gpu, shared):
    B, H, Sq, Sk, D = 128, 64, 131072, 132, 128  # 2^23 workgroups of 512
    q, k = shared(B, Sq, H, D, torch.float16), shared(B, Sk, H, D, torch.float16)
    er = 1.0 + torch.rand(Sq, Sk, generator=torch.Generator(device=gpu).manual_seed(3), device=gpu)

    def rows(q, k):
        b, _, h, _ = q.shape
        lse2 = torch.empty(b, h, Sq, dtype=torch.float32, device=gpu)
        _lib.call("dgg_attn_kf_rowlse", _lib.ptr(q), _lib.ptr(k), _lib.ptr(er), _lib.int64_array([0, 0, Sk]),
                  _lib.ptr(lse2), b, Sq, Sk, h, h, D, _lib.int64_array([*q.stride()[:3], *k.stride()[:3]]), D ** -0.5,
                  1.5, 0, 0, _lib.DGG_F16, _lib.stream_handle(gpu))
        return lse2

    want, out = rows(*_one(q, k)), rows(q, k)
    for b in range(B):  # a workgroup's place in the launch decides the order in which it adds its 132 terms
        assert (out[b] - want[0, 0]).abs().max().item() < 1e-5, f"batch {b}"
