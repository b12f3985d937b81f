"""The binding's stream argument: None is torch's current stream of the calling
thread, whatever stream or thread that is."""

import threading

import pytest
import torch

from flint_amd.flint_lib import stream_handle

pytestmark = pytest.mark.gpu


def test_none_is_the_current_stream(cuda):
    side = torch.cuda.Stream()
    for _ in range(2):   # the first call initialises, later ones ask torch directly
        assert stream_handle(None) == torch.cuda.current_stream().cuda_stream
        with torch.cuda.stream(side):
            assert stream_handle(None) == side.cuda_stream
            seen = []
            other = threading.Thread(
                target=lambda: seen.append((stream_handle(None),
                                            torch.cuda.current_stream().cuda_stream)))
            other.start()
            other.join()
            assert seen[0][0] == seen[0][1] != side.cuda_stream
        assert stream_handle(None) == torch.cuda.current_stream().cuda_stream
    assert stream_handle(side) == side.cuda_stream
    assert stream_handle(5) == 5
