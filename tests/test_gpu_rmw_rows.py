"""The full-state step's row blocks (csrc/gdnr_rmw.hip; marked `gpu`): batches
on both sides of the height rule, and V where a 64-row block does not fit,
against the oracle's step. The rows do not depend on the block, so a large
batch's first sequences equal the same ones stepped alone, bit for bit."""

from __future__ import annotations

import pytest
import torch

import gdn_replayssm_fp8_kernel as gk
from conftest import rel_l2
from gpu_helpers import np32
from oracle import gdn_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,heads,value_heads,value_dim,state", [
    (48, 16, 32, 128, torch.bfloat16), (47, 16, 32, 128, torch.bfloat16), (60, 16, 32, 128, torch.bfloat16),
    (65, 16, 32, 128, torch.float16), (130, 8, 16, 96, torch.float16),
    (128, 4, 12, 128, torch.float16), (5, 1, 3, 32, torch.bfloat16), (48, 16, 32, 128, torch.float32),
    (3, 2, 2, 96, torch.float32)])
def test_row_blocks(device, batch, heads, value_heads, value_dim, state):
    gen = torch.Generator(device=device).manual_seed(batch)
    rand = lambda *s: torch.randn(*s, generator=gen, device=device)  # noqa: E731
    unit = lambda x: torch.nn.functional.normalize(x, dim=-1)  # noqa: E731
    s0 = (0.1 * rand(batch, value_heads, value_dim, 128)).to(state)
    q, k = (unit(rand(batch, heads, 128)).bfloat16() for _ in range(2))
    v, beta = rand(batch, value_heads, value_dim).bfloat16(), torch.sigmoid(rand(batch, value_heads)).bfloat16()
    g = (-0.1 * rand(batch, value_heads).abs()).bfloat16()
    whole = s0.clone()
    out = gk.gdn_bf16_step(whole, q, k, v, g, beta)
    few = slice(0, 3)
    part = s0[few].clone()
    out_part = gk.gdn_bf16_step(part, q[few], k[few], v[few], g[few], beta[few])
    assert torch.equal(whole[few], part) and torch.equal(out[few], out_part)
    storage = {torch.bfloat16: "bf16", torch.float16: "f16", torch.float32: "f32"}[state]
    ref_out, ref_state = gdn_oracle.bf16_rmw_step(np32(s0[-2:]), *(np32(t[-2:]) for t in (q, k, v, g, beta)), storage)
    assert rel_l2(np32(out[-2:]), ref_out) <= 3e-3  # (outputs round to bf16: 1.7e-3)
    # (a state rounds to its own type; an f32 sum in another order moves few)
    assert rel_l2(np32(whole[-2:]), ref_state) <= {"bf16": 2e-4, "f16": 3e-5, "f32": 1e-6}[storage]
