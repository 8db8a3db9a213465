"""Work distribution of the forward kernels: every (sequence, head, row) is computed once, whatever order the blocks run
in and however many slices are merged.  Results against float32 math on the device (bars: tests/_util.py)."""
import ctypes
import math

import numpy as np
import pytest
import torch

import oracle
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
    (2, 64, 500),    # 512: two per CU, the second half runs backwards at head_dim 128
    (1, 65, 1000),   # 520: more than two per CU
    (2, 62, 1000),   # 992 blocks = 496 pairs: one pair per resident workgroup
    (1, 520, 130),   # 1040 blocks, two per head
    (8, 32, 300),    # 512 pairs, three blocks per head: paired at head_dim 128, heaviest first at 64, head after head at 256
    (10, 32, 500),   # 1280 blocks, four per head
])
@pytest.mark.parametrize("D", [64, 128, 256])
def test_every_causal_block_is_computed(D, B, H, S):
    q, k, v = _randn((B, H, S, D), 1, HF), _randn((B, H, S, D), 2, HF), _randn((B, H, S, D), 3, HF)
    _check(q, k, v, True)


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("B,Hq,Hk,S", [(2, 64, 16, 500), (1, 36, 4, 1000), (4, 32, 8, 1000)])   # 512, 288, 1024 blocks
def test_every_causal_block_is_computed_with_dropout_and_grouped_heads(D, B, Hq, Hk, S):
    q, k, v = _randn((B, Hq, S, D), 1, HF), _randn((B, Hk, S, D), 2, HF), _randn((B, Hk, S, D), 3, HF)
    _check(q, k, v, True)
    kw = dict(is_causal=True, dropout_p=0.25, philox_seed=3, philox_offset=8)
    mask = torch.zeros((B, Hq, S, S), dtype=HF, device=DEV)
    capi.fa_forward_dense(q, k, v, dropout_mask=mask, **kw)
    out, lse = capi.fa_forward_dense(q, k, v, **kw)
    s = q.float() @ k.float().repeat_interleave(Hq // Hk, 1).transpose(2, 3).contiguous() / math.sqrt(D)
    s.masked_fill_(torch.ones(S, S, dtype=torch.bool, device=DEV).triu(1), float("-inf"))
    want_l = torch.logsumexp(s, -1)
    keep = (math.floor(0.75 * 255) + 1) / 256
    want = (torch.exp(s - want_l[..., None]) * (mask > 0) / keep) @ v.float().repeat_interleave(Hq // Hk, 1)
    assert torch.equal(mask != 0, (s > float("-inf")))
    # the bar of the dropout tests: two units in the last place of the largest value, which the first rows' reach
    assert (out.float() - want).abs().max().item() <= 2 * 2.0 ** -11 * max(1.0, want.abs().max().item())
    assert (lse - want_l).abs().max().item() <= LSE_TOL


@pytest.mark.parametrize("D", [64, 72, 128, 256])
@pytest.mark.parametrize("Sq", [130, 300])   # 1040 rows: four wavefronts merge a row; 2400: one
def test_merge_of_slices(D, Sq):
    q, k, v = _randn((2, 4, Sq, D), 4, BF), _randn((2, 2, 4100, D), 5, BF), _randn((2, 2, 4100, D), 6, BF)
    for ns in (2, 5, 24, 64):
        _check(q, k, v, True, kernel=capi.FA_KERNEL_TILE, num_splits=ns)


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("kernel,B,Hq,Hk,Sq", [
    (capi.FA_KERNEL_TILE, 2, 4, 2, 130),      # 1040 rows: four wavefronts merge a row
    (capi.FA_KERNEL_TILE, 2, 4, 2, 300),      # 2400 rows: one
    (capi.FA_KERNEL_SPLITKV, 2, 8, 2, 2),     # 32
    (capi.FA_KERNEL_SPLITKV, 64, 32, 2, 1),   # 2048
])
def test_merge_keeps_infinities_of_the_last_slice(D, kernel, B, Hq, Hk, Sq):
    """Every row sees every key, so an infinite value of V makes its column infinite and leaves the others alone, in the
    last of the merged slices (whose partials are loaded once more in the place of slices that do not exist) too."""
    Sk = 80 * (64 if kernel == capi.FA_KERNEL_TILE else 32)  # blocks that 2, 5, 8 and 16 slices share evenly
    q, k, v = _randn((B, Hq, Sq, D), 50, HF), _randn((B, Hk, Sk, D), 51, HF), _randn((B, Hk, Sk, D), 52, HF)
    v[:, :, Sk - 7, 5] = float("inf")
    v[:, :, Sk - 3, D - 2] = float("-inf")
    whole = capi.fa_forward_dense(q, k, v, kernel=kernel, num_splits=1)[0]
    assert (whole[..., 5] == float("inf")).all() and (whole[..., D - 2] == float("-inf")).all()
    for ns in (2, 5, 8, 16):
        out = capi.fa_forward_dense(q, k, v, kernel=kernel, num_splits=ns)[0]
        assert torch.equal(out.isinf(), whole.isinf()) and torch.equal(out[whole.isinf()], whole[whole.isinf()])
        assert (out - whole).masked_fill(whole.isinf(), 0.0).abs().max().item() <= OUT_TOL[HF]  # (a NaN fails this)


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


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("B,per,ns", [
    (47, 10, 0), (48, 10, 0), (64, 10, 0), (65, 10, 0),   # 188 ... 260 units of up to 320 keys: whole (sliced at head_dim 256)
    (80, 40, 0),    # 320 of 1280: whole, four wavefronts
    (66, 64, 0),    # 264 of 2048: three slices at head_dim 128
    (126, 40, 0),   # 504 of 1280: two rounds, whole
    (124, 81, 0),   # 496 of 2592: two rounds, two slices
    (5, 50, 0),     # 20 of 1600: twelve slices
    (5, 200, 2),    # 20 of 6400: two long slices, four wavefronts
])
def test_ragged_paged_units_around_one_per_cu(D, B, per, ns):
    Hq, Hk, page = 8, 4, 32
    q = _randn((B, Hq, 1, D), 11, HF)
    kp, vp = _randn((B * per, page, Hk, D), 12, HF), _randn((B * per, page, Hk, D), 13, HF)
    g = torch.Generator(device=DEV).manual_seed(14)
    table = torch.randperm(B * per, generator=g, device=DEV).to(torch.int32).reshape(B, per)
    lens = torch.randint(1, per * page + 1, (B,), generator=g, device=DEV).to(torch.int32)
    lens[0], lens[-1] = per * page, 1
    out, lse = capi.fa_forward_paged(q, kp, vp, table, lens, num_splits=ns)
    k, v = (t[table.long()].reshape(B, per * page, Hk, D).transpose(1, 2).float() for t in (kp, vp))
    s = (q.float().reshape(B, Hk, -1, D) @ k.transpose(2, 3).contiguous()).reshape(B, Hq, -1) / math.sqrt(D)   # [B, Hq, keys]
    s.masked_fill_(torch.arange(per * page, device=DEV)[None, None, :] >= lens[:, None, None], float("-inf"))
    want_l = torch.logsumexp(s, -1)
    want = (torch.exp(s - want_l[..., None]).reshape(B, Hk, -1, per * page) @ v).reshape(B, Hq, D)
    assert (out[:, :, 0].float() - want).abs().max().item() <= OUT_TOL[HF]
    assert (lse[:, :, 0] - want_l).abs().max().item() <= LSE_TOL


def _grad_reference(q, k, v, do, causal, bias=None, keep=None, keep_p=1.0):
    """Gradients of one dense call in float64 on the CPU.  `causal`: False, True or a mask mode; `keep`: the elements that
    dropout kept, `keep_p` of them."""
    q, k, v, do = (t.double().cpu() for t in (q, k, v, do))
    g, D, Sq, Sk = q.shape[1] // k.shape[1], q.shape[3], q.shape[2], k.shape[2]
    kr, vr = k.repeat_interleave(g, 1), v.repeat_interleave(g, 1)
    s = q @ kr.transpose(2, 3) / math.sqrt(D)
    if bias is not None:
        s = s + bias.double().cpu()
    if causal:
        off = 0 if int(causal) == capi.FA_MASK_CAUSAL_TOP_LEFT else Sk - Sq
        s.masked_fill_(~(torch.arange(Sk)[None, :] <= torch.arange(Sq)[:, None] + off), float("-inf"))
    p = torch.nan_to_num(torch.softmax(s, -1))
    m = 1.0 if keep is None else keep.double().cpu() / keep_p
    dp = do @ vr.transpose(2, 3) * m
    ds = p * (dp - (p * dp).sum(-1, keepdim=True)) / math.sqrt(D)
    B, Hk = k.shape[:2]
    fold = lambda t: t.reshape(B, Hk, g, Sk, D).sum(2)
    return ds @ kr, fold(ds.transpose(2, 3) @ q), fold((p * m).transpose(2, 3) @ do)


def _check_grads(got, want, dtype):
    eps = 2.0 ** -8 if dtype == BF else 2.0 ** -11
    for name, x, w in zip(("dq", "dk", "dv"), got, want):
        x = x.double().cpu()
        assert torch.isfinite(x).all(), name
        # two units in the last place at the gradient's largest value, as for every backward test
        assert (x - w).abs().max().item() <= 2 * eps * max(w.abs().max().item(), 0.25), name


@pytest.mark.parametrize("D", [64, 72, 128, 256])
@pytest.mark.parametrize("B,Hq,Hk,Sq,Sk,causal", [
    (1, 14, 2, 130, 130, True),     # 21 and 7 steps: two slices, then one
    (1, 14, 2, 300, 500, True),     # more keys than queries, 8 (sequence, kv head, block) units
    (2, 21, 3, 500, 129, True),     # rows that see no key; a last block of one key
    (1, 12, 1, 1024, 256, False),   # equal slices
    (1, 2, 2, 1900, 64, False),     # one head's query tiles cut into slices
])
def test_sliced_key_blocks(D, B, Hq, Hk, Sq, Sk, causal):
    for dt in (BF, HF):
        q, k, v, do = (_randn(s, 20 + i, dt) for i, s in enumerate(
            [(B, Hq, Sq, D), (B, Hk, Sk, D), (B, Hk, Sk, D), (B, Hq, Sq, D)]))
        out, lse = capi.fa_forward_dense(q, k, v, is_causal=causal)
        _check_grads(capi.fa_backward_dense(do, q, k, v, out, lse, is_causal=causal), _grad_reference(q, k, v, do, causal), dt)


@pytest.mark.parametrize("D", [64, 128])
def test_sliced_key_blocks_with_a_bias(D):
    q, k, v, do = _randn((1, 14, 260, D), 30, BF), _randn((1, 2, 200, D), 31, BF), _randn((1, 2, 200, D), 32, BF), _randn((1, 14, 260, D), 33, BF)
    bias = _randn((1, 1, 260, 200), 34, BF)
    out, lse = capi.fa_forward_dense(q, k, v, bias=bias)
    _check_grads(capi.fa_backward_dense(do, q, k, v, out, lse, bias=bias)[:3], _grad_reference(q, k, v, do, False, bias), BF)


@pytest.fixture
def sliced(monkeypatch):
    """Every backward call of the test cuts key blocks: it asks for more than the two planes of its rows."""
    launch = capi._launch_bwd

    def checked(p, device):
        rows = p.total_q if p.cu_seqlens_q else p.batch * p.seqlen_q
        assert capi.lib().fa_bwd_workspace_bytes(ctypes.byref(p)) > 2 * (rows * p.heads_q * 4 + 15)
        launch(p, device)

    monkeypatch.setattr(capi, "_launch_bwd", checked)


@pytest.mark.parametrize("D", [64, 72, 128, 256])
@pytest.mark.parametrize("B,Hq,Hk,Sq,Sk", [
    (1, 14, 2, 130, 130),
    (1, 14, 2, 500, 300),    # the last rows see every key, as many as there are
    (1, 14, 2, 300, 700),    # the last keys are seen by no row
])
def test_sliced_key_blocks_top_left(sliced, D, B, Hq, Hk, Sq, Sk):
    mode = capi.FA_MASK_CAUSAL_TOP_LEFT
    q, k, v, do = (_randn(s, 80 + i, BF) for i, s in enumerate([(B, Hq, Sq, D), (B, Hk, Sk, D), (B, Hk, Sk, D), (B, Hq, Sq, D)]))
    out, lse = capi.fa_forward_dense(q, k, v, is_causal=mode)
    _check_grads(capi.fa_backward_dense(do, q, k, v, out, lse, is_causal=mode), _grad_reference(q, k, v, do, mode), BF)


@pytest.mark.parametrize("with_bias", [False, True])
@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("B,Hq,Hk,Sq,Sk,causal", [
    (1, 14, 2, 260, 260, True),
    (2, 21, 3, 400, 132, False),
    (1, 16, 1, 200, 388, capi.FA_MASK_CAUSAL_TOP_LEFT),
])
def test_sliced_key_blocks_with_dropout(sliced, D, B, Hq, Hk, Sq, Sk, causal, with_bias):
    q, k, v, do = (_randn(s, 90 + i, HF) for i, s in enumerate([(B, Hq, Sq, D), (B, Hk, Sk, D), (B, Hk, Sk, D), (B, Hq, Sq, D)]))
    bias = _randn((B, 1, Sq, Sk), 94, HF) if with_bias else None
    rng, mask = torch.zeros(2, dtype=torch.int64, device=DEV), torch.zeros((B, Hq, Sq, Sk), dtype=HF, device=DEV)
    out, lse = capi.fa_forward_dense(q, k, v, is_causal=causal, bias=bias, dropout_p=0.2, philox_seed=11, philox_offset=4,
                                     rng_out=rng, dropout_mask=mask)
    got = capi.fa_backward_dense(do, q, k, v, out, lse, is_causal=causal, bias=bias, dropout_p=0.2, rng=rng)
    keep_p = (math.floor(np.float32(1.0 - np.float32(0.2)) * np.float32(255.0)) + 1) / 256
    _check_grads(got[:3], _grad_reference(q, k, v, do, causal, bias, mask > 0, keep_p), HF)


def test_sliced_key_blocks_packed_with_dropout(sliced):
    # (no sequence of one row: its dK is exactly 0, and what a kernel gives instead is the rounding of O in delta, up to
    # heads x scale x |q| x 2^-11 x sum |dO| |O| = 7 x 0.09 x 2 x 2^-11 x 30 = 0.02 here, which the bar below does not count)
    lens, Hq, Hk, D, drop = [300, 33, 520, 64], 14, 2, 128, 0.3
    cu = np.concatenate([[0], np.cumsum(lens)]).tolist()
    q, k, v, do = (_randn(s, 100 + i, HF) for i, s in enumerate([(cu[-1], Hq, D), (cu[-1], Hk, D), (cu[-1], Hk, D), (cu[-1], Hq, D)]))
    c, rng = torch.tensor(cu, dtype=torch.int32, device=DEV), torch.zeros(2, dtype=torch.int64, device=DEV)
    out, lse = capi.fa_forward_packed(q, k, v, c, c, max(lens), max(lens), is_causal=True, dropout_p=drop, philox_seed=5,
                                      philox_offset=12, rng_out=rng)
    got = capi.fa_backward_packed(do, q, k, v, out, lse, c, c, max(lens), max(lens), is_causal=True, dropout_p=drop, rng=rng)
    row = lambda t, i: t[cu[i]:cu[i + 1]].transpose(0, 1)[None]
    for i, n in enumerate(lens):
        keep = torch.from_numpy(np.stack([oracle.dropout_keep_mask(5, 12, i * Hq + h, n, n, drop) for h in range(Hq)]))[None]
        want = _grad_reference(*(row(t, i) for t in (q, k, v, do)), True, None, keep, 1.0 - oracle.dropout_effective_p(drop))
        _check_grads([row(t, i) for t in got], want, HF)


@pytest.mark.parametrize("Hq,Hk,D", [(14, 2, 64), (14, 2, 128), (8, 1, 96)])
def test_sliced_key_blocks_packed(Hq, Hk, D):
    lens = [1, 300, 64, 0, 129, 610]
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    q, k, v, do = _randn((cu[-1], Hq, D), 40, BF), _randn((cu[-1], Hk, D), 41, BF), _randn((cu[-1], Hk, D), 42, BF), _randn((cu[-1], Hq, D), 43, BF)
    c = torch.tensor(cu, dtype=torch.int32, device=DEV)
    out, lse = capi.fa_forward_packed(q, k, v, c, c, max(lens), max(lens), is_causal=True)
    got = capi.fa_backward_packed(do, q, k, v, out, lse, c, c, max(lens), max(lens), is_causal=True)
    row = lambda t, i: t[cu[i]:cu[i + 1]].transpose(0, 1)[None]
    for i, n in enumerate(lens):
        if n:
            _check_grads([row(t, i) for t in got], _grad_reference(*(row(t, i) for t in (q, k, v, do)), True), BF)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("lens_q,lens_k", [
    ([130] * 6, [1500] * 6),                                   # more key blocks than self-attention has: room for some sequences only
    ([1, 200, 0, 64] * 20 + [900], [1, 200, 0, 64] * 20 + [900]),   # more sequences than lanes, empty ones among them
])
def test_sliced_key_blocks_packed_slots(lens_q, lens_k, causal):
    Hq, Hk, D = 28, 2, 64
    cq, ck = [0], [0]
    for n, m in zip(lens_q, lens_k):
        cq.append(cq[-1] + n)
        ck.append(ck[-1] + m)
    q, k, v, do = _randn((cq[-1], Hq, D), 44, BF), _randn((ck[-1], Hk, D), 45, BF), _randn((ck[-1], Hk, D), 46, BF), _randn((cq[-1], Hq, D), 47, BF)
    cuq, cuk = (torch.tensor(c, dtype=torch.int32, device=DEV) for c in (cq, ck))
    out, lse = capi.fa_forward_packed(q, k, v, cuq, cuk, max(lens_q), max(lens_k), is_causal=causal)
    got = capi.fa_backward_packed(do, q, k, v, out, lse, cuq, cuk, max(lens_q), max(lens_k), is_causal=causal)
    row = lambda t, c, i: t[c[i]:c[i + 1]].transpose(0, 1)[None]
    for i in (0, 1, len(lens_q) // 2 + 1, len(lens_q) - 1):
        want = _grad_reference(row(q, cq, i), row(k, ck, i), row(v, ck, i), row(do, cq, i), causal)
        _check_grads([row(got[0], cq, i), row(got[1], ck, i), row(got[2], ck, i)], want, BF)


def test_backward_without_room_for_partial_sums():
    """Less workspace than asked for, but room for the two planes: whole key blocks."""
    q, k, v, do = (_randn(s, 60 + i, BF) for i, s in enumerate([(1, 14, 300, 128), (1, 2, 500, 128), (1, 2, 500, 128), (1, 14, 300, 128)]))
    out, lse = capi.fa_forward_dense(q, k, v, is_causal=True)
    real = capi.lib()
    planes = 2 * 14 * 300 * 4

    class Short:
        def __init__(self, size):
            self.fa_bwd_workspace_bytes = lambda p: size

        def __getattr__(self, name):
            return getattr(real, name)

    try:
        assert capi.lib() is real
        capi._lib = Short(planes)
        _check_grads(capi.fa_backward_dense(do, q, k, v, out, lse, is_causal=True), _grad_reference(q, k, v, do, True), BF)
        capi._lib = Short(planes - 16)
        with pytest.raises(capi.FaFwdError):
            capi.fa_backward_dense(do, q, k, v, out, lse, is_causal=True)
    finally:
        capi._lib = real


def test_training_step_close_to_the_memory_limit():
    """The op falls back to whole key blocks where the partial sums of sliced ones do not fit."""
    import torch.nn.functional as F

    q, k, v = (_randn(s, 70 + i, BF).requires_grad_() for i, s in enumerate([(1, 28, 2048, 128), (1, 4, 2048, 128), (1, 4, 2048, 128)]))
    do = _randn((1, 28, 2048, 128), 73, BF)
    step = lambda: torch.autograd.grad(F.scaled_dot_product_attention(q, k, v, is_causal=True, enable_gqa=True), (q, k, v), do)
    want = step()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    try:   # room for the output, the gradients and the planes (36 MiB), not for 60 MiB of partial sums
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (60 << 20)) / total)
        got = step()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    for a, b in zip(got, want):
        assert torch.isfinite(a).all() and (a.float() - b.float()).abs().max().item() <= 2 * 2.0 ** -8 * max(b.abs().max().item(), 0.25)
    assert torch.equal(got[0], want[0]) and not torch.equal(got[1], want[1])   # dQ as before; dK summed in another order
