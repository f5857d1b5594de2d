"""The host extension module (csrc/gdnr_host.cpp) on the CPU: the packed step
metadata against the cache's own, and the errors of a call (the operators'
device check by argument name, accepted ranks and dtypes, the library's
status as GdnrError)."""

from __future__ import annotations

import threading
import time

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


class _Launch:
    """step()'s launch replaced by a note of the metadata it was given (with
    pageable buffers: there is no GPU to pin for)."""

    def __init__(self, monkeypatch):
        empty = torch.empty
        with torch.device("cpu"):  # (torch lists its factories at the first use of a default device)
            empty(0)
        monkeypatch.setattr(torch, "empty", lambda *shape, pin_memory=False, **kw: empty(*shape, **kw))
        monkeypatch.setattr(gk, "gdn_prep_replay_fp8", self)

    def __call__(self, mixed, a, b, a_log, dt_bias, pos, *rest, state_indices, **kw):
        self.slots, self.pos, self.valid, self.flush = state_indices, pos, rest[7], rest[8]
        return mixed


def _cpu_cache(window=4):
    return ReplaySSMCache(5, window, heads=1, value_heads=1, key_dim=128, value_dim=32, device="cpu")


def _cpu_step(cache, slots):
    rows = torch.zeros(len(slots), 1)
    return cache.step(slots, rows, rows, rows, rows[:0], rows[:0])


def test_buffers_of_other_formats_are_refused(host):
    slots, packed = np.array([1], np.int64), np.zeros(64, np.uint8)
    for fill in (np.full(4, 2.0), np.full(4, 2, np.uint64), np.zeros(4, ">i8")):
        with pytest.raises(TypeError, match="8-byte signed"):
            host.slot_metadata(fill, slots, 4, packed)
        with pytest.raises(TypeError, match="8-byte signed"):
            host.advance(fill, slots, 4)
    with pytest.raises(TypeError, match="bytes"):
        host.slot_metadata(np.zeros(4, np.int64), slots, 4, np.zeros(16, np.int32))


@pytest.mark.parametrize("dtype", [np.int32, np.int64, np.uint64, np.float64])
def test_step_takes_fills_of_any_dtype(host, monkeypatch, dtype):
    """A cache whose fill array was replaced (restored from a file, say) steps
    as metadata() says, whatever its dtype."""
    launch, cache = _Launch(monkeypatch), _cpu_cache()
    cache.fill = np.array([0, 2, 0, 3, 0, 0], dtype)
    for pos, flush in (([2, -1, 3], [0, 0, 1]), ([3, -1, 0], [1, 0, 0]), ([0, -1, 1], [0, 0, 0])):
        want = cache.metadata([1, 0, 3])
        _cpu_step(cache, [1, 0, 3])
        got = (launch.slots, launch.pos, launch.valid, launch.flush)
        assert launch.pos.tolist() == pos and launch.flush.tolist() == flush
        assert all(np.array_equal(np.asarray(x), y.astype(np.int32)) for x, y in zip(got, want))
    assert cache.fill.dtype == dtype and cache.fill.tolist() == [0, 1, 0, 2, 0, 0]


@pytest.mark.parametrize("slots", [5, np.int64(5), np.array(5), [[1, 2]]])
def test_step_refuses_slots_that_are_no_vector(host, monkeypatch, slots):
    _Launch(monkeypatch)
    with pytest.raises(ValueError, match="one-dimensional"):
        _cpu_cache().step(slots, *[torch.zeros(1, 1)] * 5)


def test_step_packs_on_the_host_under_any_default_device(host, monkeypatch):
    """torch.empty follows torch's default device; the packed metadata is host
    memory under any."""
    launch, cache = _Launch(monkeypatch), _cpu_cache()
    rows = torch.zeros(2, 1)
    with torch.device("meta"):
        cache.step([3, 0], rows, rows, rows, rows[:0], rows[:0], q_out=rows)
    assert launch.pos.tolist() == [0, -1] and launch.valid.tolist() == [1, 0]


def test_empty_lets_other_threads_run(host):
    """An allocation may wait for the device, and what the device waits for may
    need another thread: the interpreter lock is released meanwhile. (The
    allocation made slow: torch fills new memory under its deterministic mode.)"""
    like, ticks, stop = torch.empty(0, dtype=torch.bfloat16), [], threading.Event()

    def tick():
        while not stop.wait(0.001):
            ticks.append(time.perf_counter())

    thread = threading.Thread(target=tick)
    thread.start()
    torch.use_deterministic_algorithms(True)
    try:
        start = time.perf_counter()
        made = host.empty(like, (1 << 26,))
        end = time.perf_counter()
    finally:
        torch.use_deterministic_algorithms(False)
        stop.set()
        thread.join()
    assert made.shape == (1 << 26,) and made.dtype == like.dtype
    margin = 0.2 * (end - start)
    assert any(start + margin < t < end - margin for t in ticks)
