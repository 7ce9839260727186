"""The cached scratch buffers of hip_ops (CPU: the buffer logic, with a stand-in for the stream) and the
bytes that operators ask for."""

from __future__ import annotations

import threading

import pytest
import torch

from rte_amd import _lib
from rte_amd.kernels import hip_ops as H

CPU = torch.device("cpu", 0)


@pytest.fixture(autouse=True)
def _stream(monkeypatch):
    monkeypatch.setattr(H, "_WS", {})
    now = {"stream": 1}
    monkeypatch.setattr(_lib, "stream_ptr", lambda device=None: now["stream"])
    return now


def test_a_longer_buffer_does_not_show_in_the_request():
    assert H.workspace(100, CPU)[1] == 100
    at, n = H.workspace(1 << 20, CPU)
    assert n == 1 << 20
    assert H.workspace(100, CPU) == (at, 100)
    assert H.workspace(0, CPU) == (0, 0)


def test_streams_have_their_own(_stream):
    first = H.workspace(4096, CPU)[0]
    _stream["stream"] = 2
    assert H.workspace(4096, CPU)[0] != first
    _stream["stream"] = 1
    assert H.workspace(4096, CPU)[0] == first


def test_threads_on_one_stream_have_their_own():
    mine = H.workspace(4096, CPU)[0]
    other = []
    t = threading.Thread(target=lambda: other.extend(H.workspace(4096, CPU)[0] for _ in range(2)))
    t.start()
    t.join()
    assert other[0] == other[1] != mine
    assert H.workspace(4096, CPU)[0] == mine


def test_segment_sums_ask_for_no_more_partials_than_pairs():
    ask = _lib.load().rte_segment_reduce_workspace_bytes
    pairs, cols = 5000, 2048
    few_keys, many_keys = ask(pairs, 1025, cols), ask(pairs, 32768, cols)
    sort = 4 * 32768 * (pairs // 1024 + 1 + 3) + 16 * pairs  # histograms, totals, offsets; items and pairs
    assert few_keys < many_keys <= 4 * pairs * cols + sort + 4096
