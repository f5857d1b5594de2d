"""GPU parity of the long-ring full-contract path (marked `gpu`): rings of 17
to 64 tokens, which gdn_prep_replay_fp8 runs on the decode kernel's chunked
path at small batches (csrc/gdnr_decode.hip, up to 16 sequences of 32 value
heads), on the ring kernel beyond (csrc/gdnr_ring.hip), and on the fused
replay kernel (csrc/gdnr_kernels.hip) for the shapes that neither holds.

The reference's full-contract cycle (prototype/bench_gdn_full_contract.py
:225-308) over a little more than one ring with mixed ring phases, so that
every sequence flushes once and the launches mix replays and flushes. The
outputs are checked against the fp64 oracle (gdn_oracle.full_contract_decode,
which restates prototype/gdn_replay_fp8_reference.py:189-244 and the prep of
prototype/gdn_replayssm_fp8_kernel.py:453-576) to the 2e-3 rel-L2 gate; the
requantised codes to rounding-boundary flips (< 1e-3 of the codes); the
prepared query and the ring slots the prep appended to within one bf16 ulp
of the oracle's prep (the device forms them in fp32, the oracle in fp64).
The fused launch also equals the unfused pair (prep, then replay) bit for
bit at L = 64.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import gdn_replayssm_fp8_kernel as gk
import gdn_replayssm_synth as synth
from conftest import rel_l2
from gpu_helpers import codes_np, np32
from oracle import gdn_oracle

pytestmark = pytest.mark.gpu

OUT_TOL = 2e-3
CODE_FLIP_TOL = 1e-3


def _zero_rings(batch, window, shape, device):
    return [torch.zeros(batch, window, shape.heads, shape.key_dim, dtype=torch.bfloat16, device=device),
            torch.zeros(batch, window, shape.value_heads, shape.value_dim, dtype=torch.bfloat16, device=device),
            torch.zeros(batch, window, shape.value_heads, dtype=torch.bfloat16, device=device),
            torch.zeros(batch, window, shape.value_heads, dtype=torch.bfloat16, device=device)]


def _within_bf16_ulp(got, want):
    ulp = np.abs(want) * 2.0 ** -7 + 1e-30
    return bool(np.all(np.abs(got - want) <= ulp)) and float(np.mean(got != want)) < 0.01


@pytest.mark.parametrize("batch", [3, 20], ids=["decode_kernel", "ring_kernel"])
@pytest.mark.parametrize("window", [32, 64])
def test_long_ring_cycle_matches_oracle(device, window, batch):
    import gdnr_lib

    shape = synth.Shape(batch)
    # (the kernel each batch is meant to run on)
    assert (gdnr_lib.decode_plan(batch, shape.heads, shape.value_heads, shape.value_dim, window) is not None) == (batch == 3)
    gen = synth.generator(4100 + window, device)
    a_log, dt_bias = synth.gating_params(shape, gen, device)
    state = synth.warm_state(shape, 16, gen, device, a_log, dt_bias)
    steps = window + 1
    mixed, a, b = synth.raw_step_inputs(shape, steps, gen, device)
    phase = np.array([0, window // 2, window - 1] + [(5 * i) % window for i in range(batch - 3)])
    ck = gk.quantize_checkpoint(state)
    codes0, scale0 = codes_np(ck.payload).copy(), ck.scale.cpu().numpy().copy()
    q_out = torch.zeros(batch, shape.heads, shape.key_dim, dtype=torch.bfloat16, device=device)
    rings = _zero_rings(batch, window, shape, device)
    # the oracle's prep into rings of its own, step by step (the rings depend on the prep alone)
    oq = np.zeros((batch, shape.heads, shape.key_dim), np.float32)
    orings = [np.zeros(r.shape, np.float32) for r in rings]
    phase_t = torch.as_tensor(phase, dtype=torch.int32, device=device)
    outs = []
    for step in range(steps):
        fill = (phase_t + step) % window + 1
        outs.append(np32(gk.gdn_prep_replay_fp8(mixed[:, step].contiguous(), a[:, step].contiguous(),
                                                b[:, step].contiguous(), a_log, dt_bias, fill - 1, ck.payload,
                                                ck.scale, q_out, *rings, fill, fill == window)))
        gdn_oracle.prep_ring(np32(mixed[:, step]), np32(a[:, step]), np32(b[:, step]), np32(a_log), np32(dt_bias),
                             (phase + step) % window, oq, *orings)
    ref, ref_codes, _ = gdn_oracle.full_contract_decode(
        codes0, scale0, np32(mixed), np32(a), np32(b), np32(a_log), np32(dt_bias), window, shape.heads,
        shape.key_dim, shape.value_heads, shape.value_dim, phase=phase, dtype=np.float64)
    got = np.stack(outs, axis=1)
    err = rel_l2(got, ref)
    flips = float(np.mean(codes_np(ck.payload) != ref_codes))
    print(f"L={window}: output rel-L2 {err:.3e}, code flips {flips:.2e}")
    assert err <= OUT_TOL, err
    assert flips < CODE_FLIP_TOL, flips
    assert _within_bf16_ulp(np32(q_out), oq)
    for got_r, want_r in zip(rings, orings):
        assert _within_bf16_ulp(np32(got_r), want_r)


def test_long_ring_fused_equals_prep_then_replay(device):
    """gdn_prep_replay_fp8 == gdn_prep_ring + gdn_replay_fp8 bit for bit at
    L = 64: outputs, query, ring slots, codes and scales, with replays and
    flushes in the same launch and a new token outside the replayed prefix."""
    batch, window = 5, 64
    shape = synth.Shape(batch)
    gen = synth.generator(4199, device)
    a_log, dt_bias = synth.gating_params(shape, gen, device)
    state = synth.warm_state(shape, 16, gen, device, a_log, dt_bias)
    mixed, a, b = synth.raw_step_inputs(shape, 1, gen, device)
    mixed, a, b = mixed[:, 0].contiguous(), a[:, 0].contiguous(), b[:, 0].contiguous()
    _, k, v, g, beta = synth.ring_inputs(shape, window, gen, device, a_log, dt_bias)
    pos = torch.tensor([0, 17, 63, 40, 63], dtype=torch.int32, device=device)
    valid = pos + 1
    valid[3] = 20  # the new token outside the replayed prefix
    flush = torch.tensor([0, 0, 1, 0, 1], dtype=torch.bool, device=device)
    results = []
    for fused in (False, True):
        ck = gk.quantize_checkpoint(state)
        q_out = torch.zeros(batch, shape.heads, shape.key_dim, dtype=torch.bfloat16, device=device)
        rk, rv, rg, rb = k.clone(), v.clone(), g.clone(), beta.clone()
        if fused:
            out = gk.gdn_prep_replay_fp8(mixed, a, b, a_log, dt_bias, pos, ck.payload, ck.scale, q_out, rk, rv, rg,
                                         rb, valid, flush)
        else:
            gk.gdn_prep_ring(mixed, a, b, a_log, dt_bias, pos, q_out, rk, rv, rg, rb)
            out = gk.gdn_replay_fp8(ck.payload, ck.scale, q_out, rk, rv, rg, rb, valid, flush)
        results.append([out, q_out, rk, rv, rg, rb, ck.payload.view(torch.uint8), ck.scale])
    for x, y in zip(*results):
        assert torch.equal(x, y)


def test_long_ring_tiles_identical(device):
    """The requested V-tile height (block_v 32, 64 or 128) changes nothing:
    outputs, requantised codes and scales are bit-identical at L = 64, with
    replaying and flushing sequences in the same launch. (Batch 16 of this
    layer runs the decode kernel, which has no V-tiles.)"""
    from gpu_helpers import make_replay_case, run_replay

    valid = [64, 17, 33, 64, 1, 64, 50, 63, 64, 2, 40, 64, 9, 64, 31, 64]
    flush = [v == 64 for v in valid]
    results = []
    for bv in (128, 64, 32):
        case = make_replay_case(16, 64, device, seed=4300, warmup=16, valid=valid, flush=flush)
        out = run_replay(case, block_v=bv)
        results.append((out, case["ckpt"].payload.view(torch.uint8).clone(), case["ckpt"].scale.clone()))
    for other in results[1:]:
        for x, y in zip(results[0], other):
            assert torch.equal(x, y)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("batch,heads,value_heads,value_dim,window", [
    (9, 4, 8, 96, 33), (9, 4, 8, 32, 64), (43, 4, 12, 64, 64), (43, 4, 12, 64, 17)])
def test_replay_kernel_16_bit(device, batch, heads, value_heads, value_dim, window, dtype):
    """The shapes of 16-bit rings that neither the decode kernel nor the ring
    kernel holds (V = 32, 96, ...; V = 64 with an odd group past the decode
    kernel's batches): replays and flushes at fills around the 16-token
    chunks against the fp64 oracle; the fused launch and the slot-indexed one
    against prep then replay, bit for bit. Outputs 2e-3 rel-L2 over the batch;
    a single sequence's few hundred values, in which a few large ones can
    weigh most, within bf16's largest rounding, 2^-8 of each value."""
    from gpu_helpers import make_replay_case, oracle_replay, run_replay
    import gdnr_lib

    assert gdnr_lib.decode_plan(batch, heads, value_heads, value_dim, window, act=dtype) is None
    assert value_dim not in (64, 128, 256) or (value_dim == 64 and value_heads // heads % 2)  # (not the ring kernel's)
    edges = [window, 1, 16, 17, window - 1, 0]
    valid = np.array([edges[i % len(edges)] for i in range(batch)])
    flush = np.array([i % 2 == 0 for i in range(batch)])
    block_v = 64 if value_dim % 64 == 0 else 32
    case = make_replay_case(batch, window, device, seed=4400, heads=heads, value_heads=value_heads, value_dim=value_dim,
                            dtype=dtype, warmup=8, valid=valid, flush=flush, reference_dist=True)
    shape = synth.Shape(batch, heads, value_heads, value_dim=value_dim)
    gen = synth.generator(4401, device)
    a_log, dt_bias = synth.gating_params(shape, gen, device, reference_dist=True)
    mixed, a, b = (t[:, 0].contiguous() for t in synth.raw_step_inputs(shape, 1, gen, device, dtype, dtype))
    pos = torch.as_tensor(np.maximum(valid - 1, 0), dtype=torch.int32, device=device)
    slots = torch.randperm(batch, generator=torch.Generator().manual_seed(4)).to(device) + 1
    results = []
    for mode in ("pair", "fused", "slots"):
        state = [case["ckpt"].payload.view(torch.uint8).clone(), case["ckpt"].scale.clone(),
                 *(case[k].clone() for k in ("k", "v", "g", "beta"))]
        if mode == "slots":
            cache = [torch.zeros(batch + 1, *t.shape[1:], dtype=t.dtype, device=device) for t in state]
            for c, t in zip(cache, state):
                c[slots] = t
            state = cache
        payload, scale, *rings = state
        payload, q_out = payload.view(torch.float8_e4m3fn), torch.zeros_like(case["q"])
        if mode == "pair":
            gk.gdn_prep_ring(mixed, a, b, a_log, dt_bias, pos, q_out, *rings)
            out = gk.gdn_replay_fp8(payload, scale, q_out, *rings, case["valid"], case["flush"], block_v=block_v)
        else:
            out = gk.gdn_prep_replay_fp8(mixed, a, b, a_log, dt_bias, pos, payload, scale, q_out, *rings, case["valid"],
                                         case["flush"], block_v=block_v,
                                         state_indices=slots if mode == "slots" else None)
        results.append([out, q_out, *(t[slots] if mode == "slots" else t for t in (payload.view(torch.uint8), scale, *rings))])
    for other in results[1:]:
        for x, y in zip(results[0], other):
            assert torch.equal(x, y)

    out = np32(run_replay(case, block_v=block_v))
    ref, ref_codes, ref_scale = oracle_replay(case)
    codes, scale = codes_np(case["ckpt"].payload), case["ckpt"].scale.cpu().numpy()
    assert np.array_equal(codes[~flush], case["codes0"][~flush]) and np.array_equal(scale[~flush], case["scale0"][~flush])
    assert rel_l2(out, ref) <= OUT_TOL
    for i in range(batch):
        assert rel_l2(out[i], ref[i]) <= 2.0 ** -8, (i, valid[i], flush[i])
    assert np.mean(codes != ref_codes) < 1e-4
    assert np.abs(scale.view(np.int16).astype(np.int32) - ref_scale.view(np.int16).astype(np.int32)).max() <= 1


@pytest.mark.parametrize("batch,heads,value_heads,value_dim,window,dtype,tiles", [
    (43, 4, 12, 64, 40, torch.bfloat16, (64, 32)), (16, 16, 32, 128, 20, torch.float32, (64, 32))])
def test_replay_kernel_tiles_identical(device, batch, heads, value_heads, value_dim, window, dtype, tiles):
    """The replay kernel's V-tile height changes nothing, bit for bit, with
    replaying and flushing sequences in the same launch. (Batches at which the
    library lowers no tile below the requested one.)"""
    from gpu_helpers import make_replay_case, run_replay

    valid = np.array([(11 * i) % window + 1 for i in range(batch)])
    flush = valid % 3 == 0
    results = []
    for tile in tiles:
        case = make_replay_case(batch, window, device, seed=4500, heads=heads, value_heads=value_heads,
                                value_dim=value_dim, dtype=dtype, warmup=8, valid=valid, flush=flush)
        out = run_replay(case, block_v=tile)
        results.append((out, case["ckpt"].payload.view(torch.uint8).clone(), case["ckpt"].scale.clone()))
    for x, y in zip(*results):
        assert torch.equal(x, y)
