"""GPU parity of the ring kernel (csrc/gdnr_ring.hip; marked `gpu`): rings of
17 to 64 tokens with 16-bit activations past the decode kernel's batches, at
the sizes where its tiles end -- fills around every 16-token chunk, an empty
ring and partial fills that flush, rings that end inside a chunk, each of its
four workgroup shapes, and launches of more than one round, whose flushing
sequences are taken first (a few of them by two workgroups each) -- against the fp64 oracle, and the fused launch
against prep then replay bit for bit.

Tolerances: 16-bit outputs 2e-3 rel-L2 (bf16 rounds to 2^-9: 1.65e-3), codes
< 1e-4 flips (a state within f32 rounding of an e4m3 boundary: about 5e-6),
scales within one fp16 ulp."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import gdn_replayssm_fp8_kernel as gk
import gdn_replayssm_synth as synth
import gdnr_lib
from conftest import rel_l2
from gpu_helpers import codes_np, make_replay_case, np32, run_replay
from oracle import gdn_oracle

pytestmark = pytest.mark.gpu

EDGES = [0, 1, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64]
# batch, heads, value heads, V, ring, dtype
CASES = {
    "two heads a workgroup, two rounds": (50, 16, 32, 128, 64, torch.bfloat16),
    "two rounds, full rings flushing in halves": (50, 16, 32, 128, 64, torch.bfloat16),
    "one head a workgroup": (17, 16, 32, 128, 33, torch.bfloat16),
    "odd group": (43, 4, 12, 128, 17, torch.bfloat16),
    "V=256": (13, 2, 4, 256, 40, torch.bfloat16),
    "V=64": (17, 16, 32, 64, 48, torch.float16),
    "f16": (17, 16, 32, 128, 64, torch.float16),
}


@pytest.mark.parametrize("name", CASES)
def test_ring_kernel_edges(device, name):
    batch, heads, value_heads, value_dim, ring, dtype = CASES[name]
    assert gdnr_lib.decode_plan(batch, heads, value_heads, value_dim, ring, act=dtype) is None
    fills = [min(f, ring) for f in EDGES] + [ring, ring - 1]
    valid = np.array([fills[i % len(fills)] for i in range(batch)])
    flush = np.array([("halves" not in name and (i // len(fills) + i) % 2 == 0) or valid[i] == ring
                      for i in range(batch)])
    case = make_replay_case(batch, ring, device, seed=7, heads=heads, value_heads=value_heads, value_dim=value_dim,
                            dtype=dtype, warmup=8, valid=valid, flush=flush, reference_dist=True)
    block_v = min(128, value_dim)
    # the fused launch on the same rings: its new token lands at the fill's end (outside it in an empty ring)
    shape = synth.Shape(batch, heads, value_heads, value_dim=value_dim)
    gen = synth.generator(8, device)
    a_log, dt_bias = synth.gating_params(shape, gen, device, reference_dist=True)
    mixed, a, b = (t[:, 0].contiguous() for t in synth.raw_step_inputs(shape, 1, gen, device, dtype, dtype))
    pos = torch.as_tensor(np.maximum(valid - 1, 0), dtype=torch.int32, device=device)
    results = []
    for fused in (False, True):
        rings = [case[k].clone() for k in ("k", "v", "g", "beta")]
        payload, scale, q_out = case["ckpt"].payload.clone(), case["ckpt"].scale.clone(), torch.zeros_like(case["q"])
        if fused:
            out = gk.gdn_prep_replay_fp8(mixed, a, b, a_log, dt_bias, pos, payload, scale, q_out, *rings,
                                         case["valid"], case["flush"], block_v=block_v)
        else:
            gk.gdn_prep_ring(mixed, a, b, a_log, dt_bias, pos, q_out, *rings)
            out = gk.gdn_replay_fp8(payload, scale, q_out, *rings, case["valid"], case["flush"], block_v=block_v)
        results.append([out, q_out, *rings, payload.view(torch.uint8), scale])
    for x, y in zip(*results):
        assert torch.equal(x, y)

    out = run_replay(case, block_v=block_v)
    codes, scale = codes_np(case["ckpt"].payload), case["ckpt"].scale.cpu().numpy()
    kept = ~flush
    assert np.array_equal(codes[kept], case["codes0"][kept]) and np.array_equal(scale[kept], case["scale0"][kept])
    rows = np.arange(min(batch, 2 * len(fills)))  # (every edge; the oracle is slow)
    ref, ref_codes, ref_scale = gdn_oracle.replay_step(
        case["codes0"][rows], case["scale0"][rows], *(np32(case[k])[rows] for k in ("q", "k", "v", "g", "beta")),
        valid[rows], flush[rows], np.float64)
    for i in rows:
        assert rel_l2(np32(out)[i], ref[i]) <= 2e-3, (i, valid[i], flush[i])
    assert np.mean(codes[rows] != ref_codes) < 1e-4
    ulp = np.abs(scale[rows].view(np.int16).astype(np.int32) - ref_scale.view(np.int16).astype(np.int32))
    assert ulp.max() <= 1


@pytest.mark.parametrize("batch", [20, 64])
def test_ring_kernel_strided_views(device, batch):
    """Operands at the loosest strides and alignments the entry point takes
    (mixed_qkv rows that start 4 bytes past a 16-byte boundary, padded
    checkpoint rows, ring rows and scales that are slices, index vectors with
    gaps) give what contiguous copies give, bit for bit, and nothing beside
    the views is written."""
    heads, value_heads, value_dim, ring = 16, 32, 128, 40
    valid = np.array([(9 * i) % ring + 1 for i in range(batch)])
    flush = np.array([i % 4 == 1 for i in range(batch)])
    case = make_replay_case(batch, ring, device, seed=11, warmup=4, valid=valid, flush=flush, reference_dist=True)
    shape = synth.Shape(batch, heads, value_heads, value_dim=value_dim)
    gen = synth.generator(12, device)
    a_log, dt_bias = synth.gating_params(shape, gen, device, reference_dist=True)
    mixed, a, b = (t[:, 0].contiguous() for t in synth.raw_step_inputs(shape, 1, gen, device))

    def within(t, pads):
        """A copy of t as a slice of a larger buffer: pads[d] = (before, after) of dim d."""
        big = torch.full([n + lo + hi for n, (lo, hi) in zip(t.shape, pads)], 0x55, dtype=torch.uint8,
                         device=device).to(t.dtype)
        view = big[tuple(slice(lo, lo + n) for n, (lo, _) in zip(t.shape, pads))]
        return big, view.copy_(t)

    def gaps(t, step):
        big = torch.zeros(step * t.shape[0], dtype=t.dtype, device=device)
        return big[::step].copy_(t)

    payload = case["ckpt"].payload.view(torch.uint8)
    state = [payload, case["ckpt"].scale, case["k"], case["v"], case["g"], case["beta"]]
    pads = [[(0, 0), (0, 1), (0, 0), (16, 48)], [(0, 0), (0, 0), (1, 2)], [(0, 0), (3, 1), (0, 0), (0, 8)],
            [(0, 0), (0, 2), (0, 0), (8, 0)], [(0, 0), (1, 1), (1, 0)], [(1, 0), (0, 0), (3, 0)]]
    pos = case["valid"] - 1
    results = []
    for strided in (False, True):
        if strided:
            bigs, views = zip(*(within(t, p) for t, p in zip(state, pads)))
            out_big, out = within(torch.zeros(batch, value_heads, value_dim, dtype=mixed.dtype, device=device),
                                  [(0, 0), (0, 0), (1, 2)])
            q_big, q_out = within(torch.zeros_like(case["q"]), [(0, 0), (0, 1), (2, 4)])
            m, aa, bb = within(mixed, [(0, 0), (2, 4)])[1], within(a, [(0, 0), (1, 2)])[1], within(b, [(1, 1), (0, 3)])[1]
            index = [gaps(pos, 2), gaps(case["valid"], 3), gaps(case["flush"], 3)]
        else:
            views = [t.clone() for t in state]
            out, q_out = torch.zeros(batch, value_heads, value_dim, dtype=mixed.dtype, device=device), torch.zeros_like(case["q"])
            m, aa, bb, index = mixed, a, b, [pos, case["valid"], case["flush"]]
        codes, scale, *rings = views
        gk.gdn_prep_replay_fp8(m, aa, bb, a_log, dt_bias, index[0], codes.view(torch.float8_e4m3fn), scale, q_out, *rings,
                               index[1], index[2], out=out)
        results.append([out, q_out, *views])
    assert (m.data_ptr() % 16, m.stride(0) * 2 % 16) == (4, 12)
    for x, y in zip(*results):
        assert torch.equal(x, y)
    for big, t, p in [*zip(bigs, state, pads), (out_big, results[1][0], [(0, 0), (0, 0), (1, 2)]),
                      (q_big, results[1][1], [(0, 0), (0, 1), (2, 4)])]:
        inside = torch.zeros(big.shape, dtype=torch.bool, device=device)
        inside[tuple(slice(lo, lo + n) for n, (lo, _) in zip(t.shape, p))] = True
        assert bool((big[~inside] == torch.full((), 0x55, dtype=torch.uint8, device=device).to(big.dtype)).all())
