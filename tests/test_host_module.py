"""The host extension module (csrc/gdnr_host.cpp) on the CPU: the packed step
metadata against the cache's own, and the errors of a call (the operators'
device check by argument name, accepted ranks and dtypes, the library's
status as GdnrError)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import gdn_replayssm_fp8_kernel as gk
import gdnr_lib
from gdn_replayssm_cache import ReplaySSMCache


@pytest.fixture(scope="module")
def host():
    if not (gdnr_lib.LIBRARY_PATH.exists() and gdnr_lib.HOST_PATH.exists()):
        import gdnr_build

        gdnr_build.build()
    return gdnr_lib.host()


@pytest.mark.parametrize("batch", [0, 1, 7, 64])
@pytest.mark.parametrize("window", [1, 5])
def test_slot_metadata_is_the_caches(host, batch, window):
    cache = ReplaySSMCache(64, window, heads=1, value_heads=1, key_dim=128, value_dim=32, device="cpu")
    rng = np.random.RandomState(batch)
    for _ in range(7):
        slots = np.where(rng.rand(batch) < 0.2, 0, rng.permutation(64)[:batch] + 1).astype(np.int64)
        _, pos, valid, flush = cache.metadata(slots)
        packed = np.zeros(13 * batch, np.uint8)
        host.slot_metadata(cache.fill, slots, window, packed)
        ints = packed[:12 * batch].view(np.int32).reshape(3, batch)
        assert np.array_equal(ints, np.stack([slots, pos, valid])) and np.array_equal(packed[12 * batch:], flush)
        want = cache.fill.copy()
        want[slots[slots != 0]] = np.where(flush, 0, valid)[slots != 0]
        host.advance(cache.fill, slots, window)
        assert np.array_equal(cache.fill, want)


def test_slot_metadata_refuses_what_the_cache_refuses(host):
    fill = np.zeros(4, np.int64)
    for slots, text in (([1, 4], "outside"), ([-1], "outside"), ([2, 0, 2], "twice")):
        with pytest.raises(ValueError, match=text):
            host.slot_metadata(fill, np.array(slots, np.int64), 4, np.zeros(64, np.uint8))
    with pytest.raises(ValueError, match="small"):
        host.slot_metadata(fill, np.array([1, 2], np.int64), 4, np.zeros(25, np.uint8))
    with pytest.raises(TypeError, match="8-byte"):
        host.slot_metadata(fill, np.array([1], np.int32), 4, np.zeros(64, np.uint8))


def test_call_errors(host):
    x = torch.zeros(1, 1, 32, 128)
    with pytest.raises(ValueError, match="state must be a tensor on the GPU"):
        gk.quantize_checkpoint(x)
    with pytest.raises(ValueError, match="checkpoint must be a tensor on the GPU"):
        gk.gdn_replay_fp8(x, *[x] * 8)
    with pytest.raises(ValueError, match="mixed_qkv must be a tensor on the GPU"):
        gk.gdn_prep_ring("no tensor", *[x] * 10)
    codes, scale = torch.zeros(1, 1, 32, 128, dtype=torch.uint8), torch.zeros(1, 1, 1)
    with pytest.raises(ValueError, match="rank 5"):
        gdnr_lib.call("gdnr_dequantize_vblock32", [codes, scale, x[None]])
    with pytest.raises(TypeError, match="torch.float64 is not accepted"):
        gdnr_lib.call("gdnr_dequantize_vblock32", [codes, scale, x.double()])
    with pytest.raises(gdnr_lib.GdnrError, match="invalid argument: state") as error:
        gdnr_lib.call("gdnr_dequantize_vblock32", [codes, scale, x.half()])
    assert error.value.status == 1
    with pytest.raises(TypeError, match="3 tensors"):
        gdnr_lib.call("gdnr_dequantize_vblock32", [codes, scale])
