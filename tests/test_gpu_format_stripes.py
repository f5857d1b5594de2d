"""The stripe kernels of the checkpoint formats (csrc/gdnr_formats.hip; marked
`gpu`) where their layouts end: every group height and width they hold, groups
of 2 to 8 stripes, the heights and strides that stay with the generic kernels
on either side of each limit, and views whose rows are not contiguous. Codes,
scales, saturation and the read-back equal the oracle's bit for bit."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import gdn_replayssm_fp8_kernel as gk
import gdnr_lib
from gpu_helpers import np32
from oracle import gdn_oracle

pytestmark = pytest.mark.gpu

# granularity, tile size, V
CASES = [("head", 32, 32), ("head", 32, 96), ("head_int8", 32, 256), ("head", 32, 288),
         ("row", 32, 32), ("row_int8", 32, 48),
         ("tile", 2, 32), ("tile", 4, 32), ("tile_int8", 8, 64), ("tile", 16, 96), ("tile", 64, 128),
         ("tile_int8", 128, 128),
         ("vblock", 1, 32), ("vblock_int8", 2, 32), ("vblock", 4, 64), ("vblock", 8, 32), ("vblock", 24, 96),
         ("vblock", 32, 96), ("vblock_int8", 96, 96), ("vblock", 128, 256)]


def _state(device, value_dim, view):
    gen = torch.Generator(device=device).manual_seed(value_dim)
    pad = {"whole": 0, "padded rows": 4, "odd rows": 3}[view]
    x = torch.randn(3, 2, value_dim, 128 + pad, generator=gen, device=device)[..., :128]
    x[0, 1] = 0.0
    x[1, 0, 5, 7] = float("nan")
    x[1, 1, :16] *= 3.0e6                          # fp16 scales overflow
    x[2, 0, :8] *= 1.0e-30                         # and underflow
    x[2, 1, 8:24] *= 2.0e-6                        # subnormal fp16 scales
    x[2, 1, 3, 1] = float("inf")
    return x


@pytest.mark.parametrize("view", ["whole", "padded rows", "odd rows"])
@pytest.mark.parametrize("gran,tile,value_dim", CASES)
def test_stripes_match_oracle(device, gran, tile, value_dim, view):
    x = _state(device, value_dim, view)
    if (gran, tile, view) == ("vblock", 32, "odd rows"):  # (the decode path's own format takes 16-byte aligned rows)
        with pytest.raises(gdnr_lib.GdnrError, match="multiple of 16"):
            gk.quantize_checkpoint(x, gran, tile)
        return
    q = gk.quantize_checkpoint(x, gran, tile)
    with np.errstate(all="ignore"):
        ref = gdn_oracle.quantize_checkpoint(np32(x), gran, tile)
        ref_back = gdn_oracle.dequantize_checkpoint(ref)
    got = q.payload.view(torch.int8 if gran.endswith("int8") else torch.uint8).cpu().numpy()
    assert np.array_equal(got, ref.payload)
    assert np.array_equal(q.scale.cpu().numpy().view(np.uint16), ref.scale.astype(np.float16).view(np.uint16))
    assert q.saturation_fraction == pytest.approx(ref.saturation_fraction, abs=1e-12)
    assert np.array_equal(np32(gk.dequantize_checkpoint(q)), ref_back, equal_nan=True)
