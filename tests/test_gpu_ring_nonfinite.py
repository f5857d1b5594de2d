"""Infinities and NaN in a ring that the ring kernel (csrc/gdnr_ring.hip)
replays or flushes (marked `gpu`), against the fp64 oracle's recurrence and
the reference quantiser.

A value infinite in the last token leaves its row of the state +-inf, so its
vblock takes an infinite scale (finite codes 0, the row's NaN); infinite in an
earlier token, or NaN, it makes NaN of its row (the later tokens retrieve
inf - inf), and the vblock takes scale 1. No other vblock sees it.

Rows of either kind compare by NaN and infinity; everything else by the flips
and the 2e-3 rel-L2 of the finite cases (a vblock of scale 1 rounds values of
0.01 on e4m3's subnormal grid: its codes flip where the state differs by
rounding, < 1e-3 of them)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import gdnr_lib
from conftest import rel_l2
from gpu_helpers import codes_np, make_replay_case, np32, oracle_replay, run_replay

pytestmark = pytest.mark.gpu

INF, NAN = float("inf"), float("nan")
# fills: one token, chunk ends and their neighbours, two and four chunks
FILLS = [40, 33, 32, 17, 16, 1, 31, 39]


def _free(codes):
    codes = np.where(codes == 0x80, 0, codes)
    return np.where(codes == 0xFF, 0x7F, codes)


@pytest.mark.parametrize("batch,heads,value_heads,value_dim,dtype", [
    (64, 16, 32, 128, torch.bfloat16), (20, 16, 32, 128, torch.bfloat16), (20, 16, 32, 128, torch.float16),
    (9, 8, 8, 256, torch.bfloat16)])
def test_nonfinite_values(device, batch, heads, value_heads, value_dim, dtype):
    ring = 40
    assert gdnr_lib.decode_plan(batch, heads, value_heads, value_dim, ring, act=dtype) is None
    valid = np.array([FILLS[i % len(FILLS)] for i in range(batch)])
    flush = np.array([i % 16 < 8 for i in range(batch)])
    case = make_replay_case(batch, ring, device, seed=5, heads=heads, value_heads=value_heads, value_dim=value_dim,
                            dtype=dtype, warmup=8, valid=valid, flush=flush, reference_dist=True)
    v, beta = case["v"], case["beta"]
    for b, n in enumerate(valid):
        v[b, n - 1, 0, 3] = INF                    # the last token
        v[b, n - 1, 1, 40] = -INF                  # ... another head's second vblock
        v[b, n - 1, 1, 63] = INF                   # ... and once more in it
        v[b, 0, 2, 5] = INF                        # the first one (the last too where n = 1)
        v[b, n // 2, 3, 33] = NAN
        v[b, n // 2, 4, 2], v[b, n - 1, 4, 2] = -INF, INF
        v[b, n - 1, 5, 7], beta[b, n - 1, 5] = INF, 0.0  # inf beta = NaN
        v[b, n - 1, 6, 9], beta[b, n - 1, 6] = INF, -0.5
        if n < ring:
            v[b, n:, 7, 11] = INF                  # past the fill: never read
    payload = case["ckpt"].payload.view(torch.uint8)
    payload[:, 0, 3, 17] = 0x7F                    # a NaN code in an infinite row
    case["codes0"] = codes_np(case["ckpt"].payload).copy()
    out = np32(run_replay(case, block_v=min(128, value_dim)))
    with np.errstate(invalid="ignore", over="ignore"):
        ref, ref_codes, ref_scale = oracle_replay(case)
    codes, scale = codes_np(case["ckpt"].payload), case["ckpt"].scale.cpu().numpy()
    assert np.array_equal(codes[~flush], case["codes0"][~flush]) and np.array_equal(scale[~flush], case["scale0"][~flush])
    for b in range(batch):
        where = (b, valid[b], flush[b])
        assert np.array_equal(np.isnan(out[b]), np.isnan(ref[b])), where
        whole = ~np.isfinite(ref[b])
        assert np.array_equal(out[b][np.isinf(ref[b])], ref[b][np.isinf(ref[b])]), where
        assert rel_l2(out[b][~whole], ref[b][~whole]) <= 2e-3, where
        if not flush[b]:
            continue
        got, want = _free(codes[b]), _free(ref_codes[b])
        finite = np.isfinite(ref_scale[b])
        assert np.array_equal(np.isfinite(scale[b]), finite) and (~finite).any(), where
        ulp = np.abs(scale[b].view(np.int16).astype(np.int32) - ref_scale[b].view(np.int16).astype(np.int32))
        assert ulp.max() <= 1, where
        assert np.array_equal(got == 0x7F, want == 0x7F), where
        rows = np.repeat(finite, 32, axis=-1)
        assert np.array_equal(got[~rows], want[~rows]), where
        assert np.mean(got != want) < 1e-3, where


def test_infinite_query(device):
    """Of an empty ring: o = S_0 q is infinite (or NaN where a code is 0)."""
    case = make_replay_case(20, 33, device, seed=6, warmup=8, valid=np.zeros(20, np.int32), reference_dist=True)
    case["q"][:, 0, 5], case["q"][:, 3, 64] = INF, -INF
    out = np32(run_replay(case))
    with np.errstate(invalid="ignore"):
        ref, _, _ = oracle_replay(case)
    assert np.isinf(ref).any() and np.array_equal(np.isnan(out), np.isnan(ref))
    assert np.array_equal(out[np.isinf(ref)], ref[np.isinf(ref)])
    assert rel_l2(out[np.isfinite(ref)], ref[np.isfinite(ref)]) <= 2e-3
