"""``current_stream_handle`` is torch's current stream in every context a call may come from: the
default stream, a side stream, nested stream contexts, another thread and graph capture. An unpack
launched without a stream argument runs there."""
from __future__ import annotations

import threading

import pytest
import torch

from stagehand_amd.unpack import KIND_COPY_BYTES, UnpackPlan, current_stream_handle, make_descs

pytestmark = pytest.mark.gpu


def _same() -> bool:
    return current_stream_handle() == torch.cuda.current_stream().cuda_stream


def test_handle_follows_torch():
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    assert _same() and current_stream_handle() == torch.cuda.default_stream().cuda_stream
    with torch.cuda.stream(a):
        assert current_stream_handle() == a.cuda_stream and _same()
        with torch.cuda.stream(b):
            assert current_stream_handle() == b.cuda_stream
        assert current_stream_handle() == a.cuda_stream
        seen = []
        thread = threading.Thread(target=lambda: seen.append((current_stream_handle(), _same())))
        thread.start()
        thread.join()
        assert seen == [(torch.cuda.default_stream().cuda_stream, True)]  # a stream context is its thread's
    assert _same()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = current_stream_handle(), torch.cuda.current_stream().cuda_stream
        torch.zeros(1, device="cuda")
    assert captured[0] == captured[1] != torch.cuda.default_stream().cuda_stream


def test_unpack_without_a_stream_argument_is_ordered_on_the_current_stream():
    n = 64 << 20
    plan = UnpackPlan(make_descs([(KIND_COPY_BYTES, 0, 0, 1, n, 0, 0)]))
    src = torch.zeros(n, dtype=torch.uint8, device="cuda")
    dst = torch.empty_like(src)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for value in range(1, 6):
            src.fill_(value)
            plan.run(src, dst)
            assert bool((dst == value).all())
