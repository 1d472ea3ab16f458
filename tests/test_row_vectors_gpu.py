"""The wide forms of two row kernels against their one-element forms, which
other operands still take: the sum of split partials (four outputs a thread)
and the q/k norm + RoPE + cache write (four tokens a wave).  Both keep every
sum and rounding point, so the results are equal bit for bit."""
from __future__ import annotations

import pytest
import torch

DEV = "cuda"
DTYPES = pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])


def _off_by_one(t):
    """The same values at an address that is not 8-byte aligned, rows of odd stride."""
    wide = torch.empty(t.shape[0], t.shape[1] + 5, dtype=t.dtype, device=DEV)
    wide[:, 1:1 + t.shape[1]] = t
    return wide[:, 1:1 + t.shape[1]]


@pytest.mark.gpu
@DTYPES
@pytest.mark.parametrize("M", [1, 5, 16, 65, 261])
def test_reduce_of_partials_wide_equals_narrow(M, dtype):
    """N at 4, past one wave's 256 columns and past a workgroup's 1024; splits
    below and above the unrolled four; M x N on both sides of 2^20."""
    from kernels.thin_linear_fused import thin_linear, thin_linear_residual
    g = torch.Generator(device=DEV).manual_seed(M)
    for K, N, split in [(1024, 4, 2), (1000, 260, 3), (2048, 1028, 4), (1024, 4100, 7)]:
        print(f"reduce M={M} K={K} N={N} split={split} {dtype}", flush=True)
        x = torch.randn(M, K, device=DEV, generator=g).to(dtype)
        w = (torch.randn(N, K, device=DEV, generator=g) * K ** -0.5).to(dtype)
        b, res = (torch.randn(n, N, device=DEV, generator=g).to(dtype) for n in (1, M))
        cfg = (M, 16, 0, split)
        with torch.inference_mode():
            wide = thin_linear_residual(x, w, res, config=cfg)
            assert torch.equal(wide, thin_linear_residual(x, w, _off_by_one(res), config=cfg)), (K, N, "residual")
            odd = _off_by_one(torch.zeros_like(res))
            thin_linear_residual(x, w, res, out=odd, config=cfg)
            assert torch.equal(wide, odd), (K, N, "output")
            biased = thin_linear(x, w, b[0], config=cfg)
            assert torch.equal(biased, thin_linear(x, w, _off_by_one(b)[0], config=cfg)), (K, N, "bias")


@pytest.mark.gpu
@DTYPES
@pytest.mark.parametrize("M", [1, 17, 261])
def test_gated_reduce_wide_equals_narrow(M, dtype):
    """The same of the gated sum (gate and up partials, SiLU.mul): contiguous
    outputs against odd rows at an address that is not 8-byte aligned."""
    from kernels import _native
    g = torch.Generator(device=DEV).manual_seed(M)
    lib, code = _native.lib(), _native.DTYPE_CODES[dtype]
    for K, I, split in [(1024, 4, 2), (1000, 260, 3), (1024, 4100, 4)]:
        print(f"gated reduce M={M} K={K} I={I} split={split} {dtype}", flush=True)
        x = torch.randn(M, K, device=DEV, generator=g).to(dtype)
        w = (torch.randn(2 * I, K, device=DEV, generator=g) * K ** -0.5).to(dtype)
        outs = torch.zeros(M, I, dtype=dtype, device=DEV), _off_by_one(torch.zeros(M, I, dtype=dtype, device=DEV))
        ws = torch.empty(split * M * 2 * I * 4, dtype=torch.uint8, device=DEV)
        for h in outs:
            st = lib.simsd_thin_linear_silu_mul(x.data_ptr(), K, 1, w[:I].data_ptr(), K, 1, w[I:].data_ptr(), K, 1,
                                                h.data_ptr(), h.stride(0), 1, M, I, K, code, 16, 0, split, 4,
                                                ws.data_ptr(), ws.numel(), _native.stream_of(h.device))
            _native.check(st, "thin_linear_silu_mul")
        assert torch.equal(*outs) and outs[0].abs().max() > 0, (K, I)


@pytest.mark.gpu
@DTYPES
@pytest.mark.parametrize("M", [683, 1024, 1025])
def test_rope_cache_rows_equal_single_tokens(M, dtype):
    """One call over M tokens equals M / 64 calls of few: slots in aligned
    runs, runs off by one, and out of order; tail groups of 1 to 4 tokens;
    positions and slots out of range; with and without norms and second slots."""
    from kernels.attention_fused import BlockKVCache, qkv_rope_cache
    g = torch.Generator(device=DEV).manual_seed(M)
    Hq, Hkv = 16, 4
    qkv = torch.randn(M, (Hq + 2 * Hkv) * 128, device=DEV, generator=g).to(dtype)
    nw = torch.randn(128, device=DEV, generator=g).to(dtype)
    cos, sin = (torch.randn(3000, 128, device=DEV, generator=g).to(dtype) for _ in range(2))
    pos = torch.arange(M, device=DEV) + 7
    pos[5], pos[M - 1] = -1, 3000
    run = torch.arange(M, device=DEV)
    mixed = run.clone()
    mixed[8:12] = mixed[8:12].flip(0)
    mixed[20] = -1
    far = run + M + 3
    for slots, slots2, norm in [(run, None, nw), (run + 1, far, None), (mixed, far + 1, nw),
                                (torch.randperm(M, device=DEV, generator=g), None, nw), (run + M + 40, run, nw)]:
        caches = [BlockKVCache(1, Hkv, 2 * M, 32, DEV, dtype) for _ in range(2)]
        with torch.inference_mode():
            q1 = qkv_rope_cache(qkv, Hq, norm, norm, 1e-6, cos, sin, pos, slots, caches[0], 0, slots2=slots2)
            q2 = torch.cat([qkv_rope_cache(qkv[i:i + 64], Hq, norm, norm, 1e-6, cos, sin, pos[i:i + 64],
                                           slots[i:i + 64], caches[1], 0,
                                           slots2=None if slots2 is None else slots2[i:i + 64])
                            for i in range(0, M, 64)])
        assert torch.equal(caches[0].v_tiles[0], caches[1].v_tiles[0])
        assert torch.equal(q1, q2)
        assert torch.equal(caches[0].k_tiles[0], caches[1].k_tiles[0])
