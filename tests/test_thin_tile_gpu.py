"""The tile kernel of the linear layers above 8 tokens, at the edges of its
tiles: token counts around each tile's height, rows and K that leave partial
tiles and partial stages, splits along K, padded row strides, and the operands
it hands back to the row-block kernels.  Integer data, so every sum is exact
and the outputs equal the oracle's bit for bit."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from oracle import thin_linear as othin

DEV = "cuda"
TILE = (64, -1, 0, 0)          # the tile kernel at every token count it takes, its split by the sizes
NAMES = {torch.bfloat16: "bf16", torch.float16: "fp16"}


def _ints(seed, *shape, dtype, lo=-3, hi=4):
    g = torch.Generator().manual_seed(seed)
    return torch.randint(lo, hi, shape, generator=g).to(dtype).to(DEV)


def _np(t):
    return t.float().cpu().numpy()


# (K, N): partial stages (72 = 64 + 8, 1000), one stage, whole stages; rows
# short of, at and past the 64- and 128-row tiles; deep K over few rows (split)
SHAPES = [(72, 63), (64, 64), (1000, 129), (520, 517), (8192, 256), (2048, 4104)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("M", [9, 32, 33, 64, 65, 128, 129, 257, 513])
def test_tile_edges_bit_exact(M, dtype):
    from kernels.thin_linear_fused import thin_linear, thin_linear_partials, thin_linear_residual
    for K, N in SHAPES:
        x, w, b = _ints(M, M, K, dtype=dtype), _ints(K, N, K, dtype=dtype), _ints(N, N, dtype=dtype, lo=-50, hi=50)
        res = _ints(M + 1, M, N, dtype=dtype, lo=-90, hi=90)
        xs = torch.zeros(M, K + 24, dtype=dtype, device=DEV)   # padded rows, 16-byte aligned
        xs[:, :K] = x
        ws = torch.full((N, K + 8), 7.0, dtype=dtype, device=DEV)
        ws[:, :K] = w
        want = othin.linear_exact(_np(x), _np(w), dtype=NAMES[dtype])
        with torch.inference_mode():
            assert np.array_equal(_np(thin_linear(x, w, config=TILE)), want), (K, N)
            assert np.array_equal(_np(thin_linear(xs[:, :K], ws[:, :K], config=TILE)), want), (K, N, "padded rows")
            assert np.array_equal(_np(thin_linear(x, w, b, config=TILE)),
                                  othin.linear_exact(_np(x), _np(w), _np(b), NAMES[dtype])), (K, N, "bias")
            part = thin_linear_partials(x, w, config=TILE)
            assert np.array_equal(part.double().sum(0).cpu().numpy(),
                                  _np(x).astype(np.float64) @ _np(w).astype(np.float64).T), (K, N, "partials")
            got = res.clone()
            thin_linear_residual(x, w, got, out=got, config=TILE)
            assert np.array_equal(_np(got), othin.linear_residual_exact(_np(x), _np(w), _np(res), NAMES[dtype]))
            wide = torch.zeros(M, 2 * N, dtype=dtype, device=DEV)   # outputs 2 columns apart: not the tile kernel
            thin_linear_residual(x, w, res, out=wide[:, ::2], config=TILE)
            assert torch.equal(wide[:, ::2], got) and not wide[:, 1::2].any()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("M,N,K,gated,plan", [       # plan: weight rows and tokens of the tile, split
    (260, 6140, 2048, False, (128, 64, 1)), (257, 3070, 4096, True, (128, 64, 1)),
    (700, 4096, 520, False, (128, 128, 1)), (385, 3001, 1000, True, (128, 128, 1)), (260, 2048, 12288, False, (128, 128, 4)),
    (133, 3071, 4096, True, (128, 128, 2)), (257, 12288, 4096, True, (128, 128, 1)), (700, 1028, 8192, True, (128, 128, 2)),
    (640, 12300, 256, False, (256, 128, 1)), (513, 6200, 2048, True, (256, 128, 1)), (300, 4100, 12288, False, (256, 128, 4)),
    (513, 1499, 12288, True, (256, 128, 4)),
    (1025, 6141, 72, False, (128, 256, 1)), (1025, 4099, 520, True, (128, 256, 1)), (1024, 4096, 12288, False, (128, 256, 2)),
    (300, 1499, 12288, True, (128, 256, 4)), (700, 1500, 12288, True, (128, 256, 2))])
def test_prompt_tiles_vs_oracle(M, N, K, gated, plan, dtype):
    """The tiles above 64 tokens at sizes that choose them, plain and gated,
    with and without partials (summed four outputs a thread or, for odd N, one),
    partial last tiles and stages: integer data bit for bit, gated within the
    oracle's bound."""
    from kernels import _native
    out = (ctypes.c_int * 4)()
    assert _native.lib().simsd_thin_linear_plan(M, 2 * N if gated else N, K, _native.DTYPE_CODES[dtype], -1, 0, 4, out) == 0
    assert (out[0], out[1], out[3]) == plan, "the plan takes another tile here: choose a size that takes this one"
    from kernels.thin_linear_fused import thin_linear_residual, thin_linear_silu_mul
    print(f"prompt tiles M={M} N={N} K={K} gated={gated} {dtype}", flush=True)
    with torch.inference_mode():
        if not gated:
            x, w, res = _ints(M, M, K, dtype=dtype), _ints(K, N, K, dtype=dtype), _ints(N, M, N, dtype=dtype, lo=-90, hi=90)
            got = thin_linear_residual(x, w, res, config=TILE)
            assert np.array_equal(_np(got), othin.linear_residual_exact(_np(x), _np(w), _np(res), NAMES[dtype]))
            return
        g = torch.Generator(device=DEV).manual_seed(M + K)
        x = torch.randn(M, K, device=DEV, generator=g).to(dtype)
        w = (torch.randn(2 * N, K, device=DEV, generator=g) * K ** -0.5).to(dtype)
        ref = othin.gated_exact(_np(x), _np(w[:N]), _np(w[N:]), NAMES[dtype])
        got = _np(thin_linear_silu_mul(x, w[:N], w[N:], config=TILE))
        assert np.abs(got - ref).max() <= othin.tolerance(float(np.abs(ref).max()), NAMES[dtype])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("M", [9, 33, 64, 65, 200, 300])
def test_tile_gated_vs_oracle(M, dtype):
    """Gate and up rows in one tile (interleaved by 16), partial last tiles of
    either: within the reference's 16-bit bound of the exact gated product."""
    from kernels.thin_linear_fused import thin_linear_silu_mul
    for K, I in [(72, 31), (256, 64), (1000, 531), (4096, 160)]:
        g = torch.Generator(device=DEV).manual_seed(M + K)
        x = torch.randn(M, K, device=DEV, generator=g).to(dtype)
        w = (torch.randn(2 * I, K, device=DEV, generator=g) * K ** -0.5).to(dtype)
        ref = othin.gated_exact(_np(x), _np(w[:I]), _np(w[I:]), NAMES[dtype])
        with torch.inference_mode():
            got = _np(thin_linear_silu_mul(x, w[:I], w[I:], config=TILE))
        assert np.abs(got - ref).max() <= othin.tolerance(float(np.abs(ref).max()), NAMES[dtype]), (K, I)


def test_tile_split_is_sane():
    """The automatic split: 1 where the tiles fill the chip or K has few
    stages, more where a few deep tiles would leave it idle, never past 8."""
    from kernels import _native
    lib = _native.lib()
    for M in (9, 36, 64, 133, 1024):
        for rows, K in ((4096, 4096), (24576, 4096), (4096, 12288), (64, 64), (1, 8), (151936, 4096)):
            s = lib.simsd_thin_tile_split(M, rows, K, 0)
            assert s in (1, 2, 4, 8) and (s == 1 or K * 2 >= 4 * s * 128), (M, rows, K, s)
    assert lib.simsd_thin_tile_split(1024, 24576, 4096, 1) == 1
    assert lib.simsd_thin_tile_split(36, 4096, 12288, 0) > 1


# (tokens, rows, K, gated): whether the call takes the tile kernel.  Either side
# of each line, where the other kernel is slower.
LINES = [((16, 24576, 4096, False), False), ((17, 4096, 2048, False), False), ((17, 4096, 2560, False), True),
         ((32, 4096, 4096, False), True), ((32, 24576, 4096, False), False), ((36, 24576, 4096, False), True),
         ((32, 6144, 4096, False), False), ((17, 6144, 4096, False), True), ((36, 6144, 4096, False), True),
         ((32, 4096, 12288, False), True), ((32, 151936, 4096, False), True), ((28, 24576, 4096, True), False),
         ((28, 12288, 2048, True), True), ((24, 6144, 1024, True), False), ((40, 3072, 1024, True), True),
         ((49, 2048, 2048, False), False), ((64, 2048, 2048, False), False), ((65, 2048, 2048, False), True),
         ((64, 4096, 2048, True), False), ((64, 4096, 2048, False), True), ((80, 1024, 2048, False), False),
         ((133, 1024, 2048, False), True), ((256, 1024, 1024, False), False), ((512, 1024, 1024, False), True)]


def test_lines_between_tile_and_row_blocks():
    """The rule takes the kernel that was the faster on both sides of its
    lines; partials' own rule leaves 1024-row projections and the swept shapes
    below 17 tokens with the row blocks."""
    from kernels.thin_linear_fused import TILE, _launch_config, _partials_config
    for (M, rows, K, gated), tile in LINES:
        got = _launch_config(M, rows, K, 2, None, None, gated=gated)
        assert (got[0] == TILE) == tile, (M, rows, K, gated, got)
        assert _launch_config(M, rows, K, 2, None, None, vec=lambda: False, gated=gated)[0] != TILE
        assert _launch_config(M, rows, K, 4, None, None, gated=gated)[0] != TILE
    for M, rows, K, tile in [(9, 4096, 12288, True), (48, 4096, 4096, True), (16, 6144, 4096, False), (17, 6144, 4096, True),
                             (16, 2048, 2048, False), (17, 2048, 2048, True), (9, 4096, 2048, False), (32, 1024, 4096, False)]:
        cfg = _partials_config(M, rows, K)
        assert (cfg is not None and cfg[1] == TILE) == tile, (M, rows, K, cfg)


def test_split_follows_who_sums_the_partials():
    """A wide, deep verify projection splits K although the call sums its own
    partials; one whose tiles fill the chip does not; a short one splits only
    where its consumer sums them, without a launch for it."""
    from kernels import _native
    split = _native.lib().simsd_thin_tile_split
    assert split(17, 6144, 4096, 0) == 4 and split(32, 8192, 2560, 0) == 2
    assert split(28, 24576, 4096, 0) == 1 and split(36, 24576, 4096, 0) == 1
    assert split(17, 6144, 1024, 0) == 1 and split(17, 6144, 1024, 1) == 2


def test_negative_split_is_refused():
    """A negative SPLIT_K raises before any launch, with BLOCK_N TILE as without."""
    from kernels.thin_linear_fused import TILE, _launch_config
    for block_n in (TILE, 16):
        with pytest.raises(ValueError, match="SPLIT_K"):
            _launch_config(36, 4096, 4096, 2, (64, block_n, 0, -2), None)
    assert _launch_config(36, 4096, 4096, 2, (64, TILE, 0, 0), None)[2] == 4


@pytest.mark.parametrize("M", [4, 16, 17, 32, 36, 48, 64, 133, 1024])
def test_pick_config_is_what_runs(M):
    """pick_config's geometry and split are those the calls take, and passing
    it back as the config gives the same call."""
    from kernels.thin_linear_fused import TILE, _launch_config, pick_config
    for K, rows in ((4096, 6144), (4096, 4096), (4096, 24576), (12288, 4096), (2048, 2048), (3000, 5000)):
        for gated in (False, True):
            cfg, runs = pick_config(M, rows, K, gated=gated), _launch_config(M, rows, K, 2, None, None, gated=gated)
            assert (cfg[1] == TILE) == (runs[0] == TILE) and cfg[3] == runs[2], (M, rows, K, gated)
            assert _launch_config(M, rows, K, 2, cfg, runs[3], gated=gated) == runs, (M, rows, K, gated)
        assert pick_config(M, rows, K, 4)[1] != TILE
