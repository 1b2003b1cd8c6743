"""The stream that operations launch on is torch's current one: the default, a side stream, and each thread's own."""
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu


def test_operations_follow_the_current_stream():
    from hydrainfer_amd import _lib
    handle = lambda: torch.cuda.current_stream().cuda_stream
    assert _lib.current_stream() == handle()
    side, seen = torch.cuda.Stream(), []
    with torch.cuda.stream(side):
        assert _lib.current_stream() == side.cuda_stream == handle()
        thread = threading.Thread(target=lambda: seen.append((_lib.current_stream(), handle())))
        thread.start()
        thread.join()
    assert seen[0][0] == seen[0][1] != side.cuda_stream
    assert _lib.current_stream() == handle() != side.cuda_stream
