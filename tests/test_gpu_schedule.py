"""Work distribution of the forward kernels: every (sequence, head, row) is computed once, whatever order the blocks run
in and however many slices are merged.  Results against float32 math on the device (bars: tests/_util.py)."""
import math

import pytest
import torch

from tests._util import LSE_TOL, OUT_TOL
from torch_mlu_amd import capi

pytestmark = pytest.mark.gpu
DEV = "cuda"
BF, HF = torch.bfloat16, torch.float16


def _randn(shape, seed, dtype):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(shape, generator=g, device=DEV) * 0.5).to(dtype)


def _check(q, k, v, causal, **kw):
    out, lse = capi.fa_forward_dense(q, k, v, is_causal=causal, **kw)
    g = q.shape[1] // k.shape[1]
    kf, vf = k.float().repeat_interleave(g, 1), v.float().repeat_interleave(g, 1)
    s = q.float() @ kf.transpose(2, 3).contiguous() / math.sqrt(q.shape[3])
    if causal:
        Sq, Sk = s.shape[2:]
        keep = torch.arange(Sk, device=DEV)[None, :] <= torch.arange(Sq, device=DEV)[:, None] + Sk - Sq
        s.masked_fill_(~keep, float("-inf"))
    want_l = torch.logsumexp(s, -1)
    want = torch.exp(s - want_l[..., None]) @ vf
    assert (out.float() - want).abs().max().item() <= OUT_TOL[q.dtype]
    assert (lse - want_l).abs().max().item() <= LSE_TOL


@pytest.mark.parametrize("B,H,S", [
    (1, 33, 1024),   # 264 blocks: a few more than one per CU, heads do not divide 256
    (1, 64, 640),    # 320
    (2, 64, 500),    # 512: two per CU, the second half runs backwards
    (1, 65, 1000),   # 520: more than two per CU
    (2, 62, 1000),   # 992 blocks = 496 pairs: one pair per resident workgroup
    (1, 520, 130),   # 1040 blocks, two per head
])
def test_every_causal_block_is_computed(B, H, S):
    q, k, v = _randn((B, H, S, 64), 1, HF), _randn((B, H, S, 64), 2, HF), _randn((B, H, S, 64), 3, HF)
    _check(q, k, v, True)


@pytest.mark.parametrize("D", [64, 72, 128, 256])
@pytest.mark.parametrize("Sq", [130, 300])   # 1040 rows: four wavefronts merge a row; 2400: one
def test_merge_of_slices(D, Sq):
    q, k, v = _randn((2, 4, Sq, D), 4, BF), _randn((2, 2, 4100, D), 5, BF), _randn((2, 2, 4100, D), 6, BF)
    for ns in (2, 5, 24, 64):
        _check(q, k, v, True, kernel=capi.FA_KERNEL_TILE, num_splits=ns)


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("used", [None, 31, 32, 33, 127, 128, 129, 255, 257, 1000])
def test_decode_slices_around_the_blocks_of_a_wavefront(D, used):
    """Slices of 0, 1, 2 and more 32-row blocks per wavefront, four wavefronts a workgroup (equal lengths) and two
    (`seqused_k`)."""
    B, Hq, Hk, Sk = 3, 6, 2, 1000
    q, k, v = _randn((B, Hq, 1, D), 7, BF), _randn((B, Hk, Sk, D), 8, BF), _randn((B, Hk, Sk, D), 9, BF)
    n = used or Sk
    lens = None if used is None else torch.full((B,), used, dtype=torch.int32, device=DEV)
    for ns in (0, 1, 2, 7):
        out, lse = capi.fa_forward_dense(q, k, v, kernel=capi.FA_KERNEL_SPLITKV, num_splits=ns, seqused_k=lens)
        s = q.float() @ k[:, :, :n].float().repeat_interleave(3, 1).transpose(2, 3).contiguous() / math.sqrt(D)
        want_l = torch.logsumexp(s, -1)
        want = torch.exp(s - want_l[..., None]) @ v[:, :, :n].float().repeat_interleave(3, 1)
        assert (out.float() - want).abs().max().item() <= OUT_TOL[BF]
        assert (lse - want_l).abs().max().item() <= LSE_TOL
