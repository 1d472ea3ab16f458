"""The many-row attention form (more than 32 query rows per KV head) at the
edges of its tiles: row counts around its blocks and workgroups, lengths around
its 16-key tiles, 64-key steps and 128-key rounds, one chunk and several, odd
GQA ratios, masks whose steps are empty, full or mixed (bytes other than 1
among them), a device-side length inside a step over slots that hold Inf and
NaN, a negative scale and strided queries -- against the fp64 oracle within the
reference's bf16 bound, 2^-7 max|ref| + 1e-3."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import attention as oatt

pytestmark = pytest.mark.gpu
DEV = "cuda"
D = 128


def _rnd(seed, *shape, dtype=torch.bfloat16):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(*shape, generator=g, device=DEV).to(dtype)


def _check(M, Hq, Hkv, L, cap=None, mask=None, dtype=torch.bfloat16, scale=None, dev_len=None, q=None):
    from kernels.attention_fused import BlockKVCache, block_attention
    print(f"attn tile M={M} Hq={Hq} Hkv={Hkv} L={L} dev_len={dev_len} masked={mask is not None}", flush=True)
    cache = BlockKVCache(1, Hkv, cap or L, 32, DEV, dtype)
    n = L if dev_len is None else dev_len
    k, v = _rnd(1, Hkv, n, D, dtype=dtype), _rnd(2, Hkv, n, D, dtype=dtype)
    cache.store(0, k, v)
    if cache.full_len > n:                         # stale slots: nothing of them may reach the output
        bad = torch.full((Hkv, cache.full_len - n, D), float("inf"), device=DEV, dtype=dtype)
        bad[:, 1::2] = float("nan")
        cache.store(0, bad, bad, start=n)
    q = _rnd(3, M, Hq, D, dtype=dtype) if q is None else q
    if mask is not None:
        mask = torch.nn.functional.pad(mask, (0, cache.full_len - mask.shape[1]))
    dl = None if dev_len is None else torch.tensor([dev_len], device=DEV)
    with torch.inference_mode():
        out = block_attention(q, cache, 0, mask, valid_len=L, valid_len_dev=dl, scale=scale)
        again = block_attention(q, cache, 0, mask, valid_len=L, valid_len_dev=dl, scale=scale)
    assert torch.equal(out, again)
    ref = oatt.attention(q.float().cpu().numpy(), k.float().cpu().numpy(), v.float().cpu().numpy(),
                         None if mask is None else (mask[:, :n] != 0).cpu().numpy(), D ** -0.5 if scale is None else scale)
    got = out.view(M, Hq, D).float().cpu().numpy()
    err = float(np.abs(got - ref).max())
    assert err <= 2 ** -7 * float(np.abs(ref).max()) + 1e-3, err
    return got


@pytest.mark.parametrize("M,Hq,Hkv", [(33, 2, 2), (17, 4, 2), (11, 6, 2), (9, 8, 2), (64, 1, 1), (65, 2, 1), (13, 15, 3),
                                      (129, 4, 4), (300, 4, 1)])
def test_rows_and_ratios(M, Hq, Hkv):
    for L in (1, 16, 65, 128, 200):
        _check(M, Hq, Hkv, L)


@pytest.mark.parametrize("L", [15, 31, 33, 63, 64, 127, 129, 255, 257, 385, 1000, 2500, 5000])
def test_lengths(L):
    for M, Hq, Hkv in ((36, 4, 1), (20, 16, 8), (150, 4, 2)):
        _check(M, Hq, Hkv, L, cap=L + 70)


@pytest.mark.parametrize("L,dev_len", [(400, 1), (400, 129), (400, 250), (700, 383), (3000, 700), (3000, 2999)])
def test_device_length(L, dev_len):
    mask = torch.rand(40, L, device=DEV, generator=torch.Generator(device=DEV).manual_seed(4)) < 0.7
    mask[:, 0] = True
    _check(40, 8, 2, L, mask=mask, dev_len=dev_len)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_masks(dtype):
    M, L = 200, 333
    blk = torch.arange(M, device=DEV) // 4
    causal = torch.zeros(M, L, dtype=torch.bool, device=DEV)
    causal[:, :133] = True                                    # a context every row sees
    causal[:, 133:] = blk[None, :] <= blk[:, None]
    _check(M, 4, 2, L, mask=causal, dtype=dtype)
    late = torch.zeros(M, L, dtype=torch.uint8, device=DEV)   # rows that see nothing, or one late slot
    late[::3, L - 1] = 255
    late[1::3, 70:200] = 2
    got = _check(M, 4, 2, L, mask=late, dtype=dtype)
    assert np.all(got[2::3] == 0)


def test_scale_and_strides():
    _check(40, 8, 4, 300, scale=-0.07)
    wide = _rnd(5, 40, 24, 2 * D)
    _check(40, 8, 4, 300, q=wide[:, 3:11, :D])                # strided rows and heads
    _check(40, 8, 4, 300, q=_rnd(6, 40, D, 8).transpose(1, 2))   # copied by the entry point


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("M,Hq,Hkv,L", [(36, 32, 8, 1000), (20, 16, 2, 4000), (200, 8, 2, 200), (150, 4, 1, 12000)])
def test_weights_keep_32_bits(M, Hq, Hkv, L, dtype):
    """The softmax weights and their sums keep 32-bit precision: the result is
    as near the fp64 one as its own rounding to 16 bits lets it be (2-norms;
    weights rounded to 16 bits would add a quarter).  5% is for fp32 sums and
    ties that round the other way."""
    from kernels.attention_fused import BlockKVCache, block_attention
    print(f"attn weights M={M} Hq={Hq} Hkv={Hkv} L={L} {dtype}", flush=True)
    cache = BlockKVCache(1, Hkv, L, 32, DEV, dtype)
    k, v, q = _rnd(1, Hkv, L, D, dtype=dtype), _rnd(2, Hkv, L, D, dtype=dtype), _rnd(3, M, Hq, D, dtype=dtype)
    cache.store(0, k, v)
    with torch.inference_mode():
        got = block_attention(q, cache, 0, None, valid_len=L).view(M, Hq, D).double().cpu()
    ref = torch.from_numpy(np.asarray(oatt.attention(q.float().cpu().numpy(), k.float().cpu().numpy(),
                                                     v.float().cpu().numpy(), None, D ** -0.5), dtype=np.float64))
    rounding = float((ref.to(dtype).double() - ref).norm())
    assert float((got - ref).norm()) <= 1.05 * rounding


def _bytes(M, Hq, Hkv, L):
    from kernels import _native
    return _native.lib().simsd_block_attention_workspace_bytes(M, Hq, Hkv, L)


def _chunked(M, Hq, Hkv, n):
    """Workspace of n chunks of keys: counters, partials, and their maxima and sums."""
    up = lambda b: -(-b // 256) * 256
    rows = -(-M * Hq // Hkv // 16) * 16
    return up(Hkv * 4) + up(Hkv * n * rows * D * 4) + up(Hkv * n * rows * 8)


# 3 to 8 row blocks over more than one round of keys and few chunks
SHORT = [(5, 16, 2, 505), (9, 32, 8, 509), (36, 8, 8, 540), (64, 8, 8, 264), (16, 16, 2, 216), (100, 8, 8, 300), (24, 16, 8, 248)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("M,Hq,Hkv,L", SHORT)
def test_short_contexts_take_direct_chunks(M, Hq, Hkv, L, dtype):
    """33 to 128 rows over short contexts: 64-key chunks, a wave a row block,
    with masks (rows that see nothing among them) and device-side lengths
    inside a step, inside a chunk and at its end."""
    assert _bytes(M, Hq, Hkv, L) == _chunked(M, Hq, Hkv, -(-L // 64))
    assert _bytes(M, Hq, Hkv, 8000) < _chunked(M, Hq, Hkv, 8000 // 64)      # longer: chunks of whole rounds
    mask = torch.rand(M, L, device=DEV, generator=torch.Generator(device=DEV).manual_seed(4)) < 0.6
    mask[1] = False
    _check(M, Hq, Hkv, L, dtype=dtype)
    _check(M, Hq, Hkv, L, mask=mask, dtype=dtype)
    for dev_len in (1, 64, 101, 128, L - 1):
        _check(M, Hq, Hkv, L, cap=L + 64, mask=mask, dev_len=dev_len, dtype=dtype)
