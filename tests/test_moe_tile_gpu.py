"""Grouped projections over runs of tiles (experts holding more slots than a
16-slot tile on average) and the wide combine, at the edges of the runs: slot
counts per expert around 16, 64 and 128, empty experts, one expert with
everything, invalid ids, ragged H and I, a shared expert with a partial run,
more slots than one scatter span -- equal bit for bit to the oracle and to the
single-tile kernels, on data whose every step is exact: gates are 0 or at least
32, where silu(g) is 0 or rounds to g, and the sums are of small integers."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import moe as omoe

DEV = "cuda"


def _ints(g, *shape, lo=-2, hi=3, dtype=torch.bfloat16):
    return torch.randint(lo, hi, shape, generator=g).to(dtype).to(DEV)


def _sparse(g, *shape, values, dtype):
    """One entry in eight from ``values``, the others zero: the steps' sums then
    stay below fp16's 65504 (the largest |y| of these sizes is 1.3e4)."""
    pick = torch.tensor(values)[torch.randint(0, len(values), shape, generator=g)]
    return (pick * (torch.rand(shape, generator=g) < 0.125)).to(dtype).to(DEV)


def _np(t):
    return t.float().cpu().numpy().astype(np.float64)


def _ids(pattern, T, k, E, g):
    if pattern == "one":
        ids = torch.zeros(T, k, dtype=torch.int64)
        ids[:, 1:] = torch.arange(1, k)[None]
    elif pattern == "edges":               # experts of 16, 17, 64, 65, 128 and 129 slots, the rest spread
        flat = torch.cat([torch.full((n,), e, dtype=torch.int64) for e, n in enumerate((16, 17, 64, 65, 128, 129))])
        flat = torch.cat([flat, torch.randint(7, E, (T * k - flat.numel(),), generator=g)])
        ids = flat[torch.randperm(T * k, generator=g)].view(T, k)
    else:
        ids = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)])
    if pattern == "invalid":
        ids[::7, 0] = -1
        ids[3::11, -1] = E + 2
    return ids.to(DEV)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("pattern,T,k,E,H,I,Is", [("edges", 200, 4, 16, 128, 64, 64), ("one", 130, 3, 8, 72, 40, 0),
                                                  ("spread", 64, 2, 4, 264, 96, 32), ("spread", 333, 8, 64, 136, 72, 40),
                                                  ("invalid", 150, 4, 8, 64, 24, 24), ("spread", 1000, 8, 16, 64, 32, 0),
                                                  ("spread", 77, 1, 3, 128, 33 * 8, 8), ("spread", 96, 8, 64, 64, 1280, 0)])
def test_runs_equal_oracle_and_single_tiles(pattern, T, k, E, H, I, Is, dtype):
    from kernels.moe_dispatch_fused import _align, _grouped_ffn, _num_tiles
    print(f"moe runs {pattern} T={T} k={k} E={E} H={H} I={I} Is={Is} {dtype}", flush=True)
    g = torch.Generator().manual_seed(T + E)
    ids = _ids(pattern, T, k, E, g)
    assert T * k >= (11 if E * I >= 10 * 256 * 32 else 18) * E     # the rule's side with runs
    x = _sparse(g, T, H, values=[1.0], dtype=dtype)
    wg, wu, wd = (_sparse(g, E, I, H, values=[32.0], dtype=dtype), _ints(g, E, I, H, lo=-1, hi=2, dtype=dtype),
                  _sparse(g, E, H, I, values=[-1.0, 1.0], dtype=dtype))
    tw = (torch.randint(1, 257, (T, k), generator=g) / 256).to(DEV)   # products with the y (multiples of 32) exact
    shared = ((_sparse(g, Is, H, values=[32.0], dtype=dtype), _ints(g, Is, H, lo=-1, hi=2, dtype=dtype),
               _sparse(g, H, Is, values=[-1.0, 1.0], dtype=dtype)) if Is else None)
    slots, te = _align(ids, E, _num_tiles(T * k, E))
    with torch.inference_mode():
        got = _grouped_ffn(x, ids, tw, wg, wu, wd, slots, te, shared=shared)
        # the same step over a stack of many more (never picked) experts: below the rule's line, single tiles
        n = T * k // 10 + 1
        pad = [torch.zeros(n, *w.shape[1:], dtype=dtype, device=DEV) for w in (wg, wu, wd)]
        big = [torch.cat((w, p)) for w, p in zip((wg, wu, wd), pad)]
        ids1 = torch.where((ids >= 0) & (ids < E), ids, torch.full_like(ids, -1))
        te1 = torch.where(te == E, torch.full_like(te, E + n), te)
        one = _grouped_ffn(x, ids1, tw, *big, slots, te1, shared=shared)
        wide = torch.zeros(T, 2 * H, dtype=dtype, device=DEV)    # outputs 2 apart: the narrow combine
        _grouped_ffn(x, ids, tw, wg, wu, wd, slots, te, shared=shared, out=wide[:, ::2])
    ref = omoe.dispatch_grouped(_np(x), ids.cpu().numpy(), _np(tw), _np(wg), _np(wu), _np(wd),
                                dtype={torch.bfloat16: "bf16", torch.float16: "fp16"}[dtype],
                                shared=None if shared is None else tuple(_np(w) for w in shared))
    assert np.abs(ref).max() > 32 and np.isfinite(ref).all()
    assert np.array_equal(_np(got), ref)
    assert torch.equal(one, got)
    assert torch.equal(wide[:, ::2], got) and not wide[:, 1::2].any()


@pytest.mark.gpu
@pytest.mark.parametrize("M,E", [(1, 1), (63, 5), (64, 7), (1023, 256), (1025, 1000), (8008, 256), (8192, 1024), (8192, 2)])
def test_align_spans(M, E):
    """The stable scatter over 16 spans of slots: the tables equal the
    oracle's counting sort."""
    from kernels.moe_dispatch_fused import moe_align
    g = torch.Generator().manual_seed(M)
    ids = torch.randint(-1, E + 1, (M, 1), generator=g)
    al = moe_align(ids.to(DEV), E)
    flat = ids.view(-1)
    keep = (flat >= 0) & (flat < E)
    order = torch.sort(torch.where(keep, flat, torch.tensor(E)), stable=True).indices
    assert torch.equal(al.perm.cpu().long(), order)
    counts = torch.bincount(flat[keep], minlength=E)
    assert torch.equal(al.counts.cpu().long(), counts)
    slots = al.slots.cpu()
    assert torch.equal(slots[slots >= 0].long(), order[:int(keep.sum())])
