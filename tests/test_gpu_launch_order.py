"""Launches that take their sequences in another order than the batch's
(marked `gpu`): the ring kernel's, flushing sequences first and a few of them
by two workgroups each (csrc/gdnr_ring.hip, past one round of workgroups), and
the decode kernel's large launches, which swap late flushes forward
(csrc/gdnr_decode.hip). Each sequence must be stepped once, as in a launch
that keeps the batch's order: outputs, query, ring rows, codes and scales bit
for bit, replayed, fused, and through slots.

The reference is the same kernel on the same sequences in launches that do not
reorder: of one round of workgroups, or (the ring kernel's two-wave shape,
which never runs in one round) of more sequences than it orders. Flushing
sequences sit on both sides of every 64-sequence word of the kernel's ballots."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import gdn_replayssm_fp8_kernel as gk
import gdn_replayssm_synth as synth
import gdnr_lib
from gpu_helpers import make_replay_case

pytestmark = pytest.mark.gpu

# ring-kernel shapes: heads, value heads, V, dtype, sequences of a reference
# launch, batches to check (B * H * head groups past 3 workgroups per compute unit)
RING = 33
SHAPES = {
    "two waves a head": (16, 32, 128, torch.bfloat16, 264, (65, 130, 256, 257)),
    "four waves a head": (16, 32, 128, torch.float16, 20, (25, 40)),
    "odd group": (4, 12, 128, torch.bfloat16, 60, (130,)),
    "V=256": (4, 8, 256, torch.bfloat16, 60, (200,)),
    "V=64": (16, 32, 64, torch.bfloat16, 40, (80,)),
}


def _case(device, batch, ring, heads, value_heads, value_dim, dtype):
    """A case of `batch` sequences at all fills, with the next token's inputs."""
    valid = np.array([(7 * i) % ring + 1 for i in range(batch)])
    case = make_replay_case(batch, ring, device, seed=9, heads=heads, value_heads=value_heads, value_dim=value_dim,
                            dtype=dtype, warmup=2, valid=valid, reference_dist=True)
    shape = synth.Shape(batch, heads, value_heads, value_dim=value_dim)
    gen = synth.generator(10, device)
    a_log, dt_bias = synth.gating_params(shape, gen, device, reference_dist=True)
    mixed, a, b = (t[:, 0].contiguous() for t in synth.raw_step_inputs(shape, 1, gen, device, dtype, dtype))
    case.pop("state")
    case.update(mixed=mixed, a=a, b=b, a_log=a_log, dt_bias=dt_bias)
    return case


def _run(case, rows, flush, mode, block_v):
    """One launch of the case's sequences `rows`; what it wrote, row by row."""
    at = torch.as_tensor(rows, device=case["q"].device)
    take = lambda t: t[at].contiguous()  # noqa: E731
    state = [take(case["ckpt"].payload.view(torch.uint8)), take(case["ckpt"].scale)] + [take(case[k]) for k in ("k", "v", "g", "beta")]
    q, valid = take(case["q"]), take(case["valid"])
    flush = torch.as_tensor(flush, dtype=torch.bool, device=q.device)
    slots = None
    if mode == "slots":  # the same rows scattered over a cache (slot 0 the null slot)
        slots = torch.randperm(len(rows), generator=torch.Generator().manual_seed(3)).to(q.device) + 1
        cache = [torch.zeros(len(rows) + 1, *t.shape[1:], dtype=t.dtype, device=t.device) for t in state]
        for c, t in zip(cache, state):
            c[slots] = t
        state = cache
    payload, scale, *rings = state
    payload = payload.view(torch.float8_e4m3fn)
    if mode == "replay":
        out = gk.gdn_replay_fp8(payload, scale, q, *rings, valid, flush, block_v=block_v)
    else:
        q = torch.zeros_like(q)
        out = gk.gdn_prep_replay_fp8(take(case["mixed"]), take(case["a"]), take(case["b"]), case["a_log"],
                                     case["dt_bias"], valid - 1, payload, scale, q, *rings, valid, flush,
                                     block_v=block_v, state_indices=slots)
    state = [payload.view(torch.uint8), scale, *rings]
    if mode == "slots":
        state = [t[slots] for t in state]
    return [out, q, *state]


def _check(case, batches, reference, mode, block_v, counts):
    total = max(reference, *batches)
    groups = [np.arange(lo, min(lo + reference, total)) for lo in range(0, total, reference)]
    want = []
    for value in (False, True):  # every sequence replayed, and every one flushed
        parts = [_run(case, g, [value] * len(g), "replay" if mode == "replay" else "fused", block_v) for g in groups]
        want.append([torch.cat(ts) for ts in zip(*parts)])
    for batch in batches:
        edges = [p for w in range(0, batch, 64) for p in (w + 63, w, w + 64, w + 30) if p < batch]
        order = list(dict.fromkeys(edges + list(range(batch))))  # (flushing sequences from the words' edges on)
        rows = np.random.RandomState(batch).permutation(total)[:batch]
        for count in counts:
            if count > batch:
                continue
            flush = np.zeros(batch, bool)
            flush[order[:count]] = True
            got = _run(case, rows, flush, mode, block_v)
            for name, x, *y in zip(("out", "q", "codes", "scale", "k", "v", "g", "beta"), got, *want):
                at = torch.as_tensor(rows, device=x.device)
                f = torch.as_tensor(flush, device=x.device)
                expect = torch.where(f.view(-1, *[1] * (x.dim() - 1)), y[1][at], y[0][at])
                assert torch.equal(x, expect), (batch, count, name, torch.nonzero((x != expect).flatten(1).any(1)).flatten().tolist())


@pytest.mark.parametrize("mode", ["replay", "fused", "slots"])
@pytest.mark.parametrize("shape", SHAPES)
def test_ring_kernel_order(device, shape, mode):
    heads, value_heads, value_dim, dtype, reference, batches = SHAPES[shape]
    for batch in (reference, *batches):
        assert gdnr_lib.decode_plan(batch, heads, value_heads, value_dim, RING, act=dtype) is None
    case = _case(device, max(reference, *batches), RING, heads, value_heads, value_dim, dtype)
    # no flush, one, as many as get two workgroups each, one more, many, all
    _check(case, batches, reference, mode, min(128, value_dim), (0, 1, 8, 9, 24, 256))


@pytest.mark.parametrize("mode", ["replay", "fused", "slots"])
@pytest.mark.parametrize("value_heads,value_dim", [(32, 128), (32, 64), (16, 256)])
def test_decode_kernel_swap(device, value_heads, value_dim, mode):
    """B = 259 and 300 (16 units and more per compute unit) against launches
    of 100 sequences, which keep the batch's order."""
    ring = 5
    case = _case(device, 300, ring, 16, value_heads, value_dim, torch.bfloat16)
    assert gdnr_lib.decode_plan(259, 16, value_heads, value_dim, ring)["units"] == 1
    _check(case, (259, 300), 100, mode, min(128, value_dim), (0, 1, 33, 200))
