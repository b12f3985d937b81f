"""A forked child's first call asks torch for its stream again: torch refuses it
where the parent has used the GPU, and the binding must not go round that."""

import os

from flint_amd import flint_lib


def test_a_forked_child_asks_torch_again(monkeypatch):
    monkeypatch.setattr(flint_lib, "_current_stream", lambda: 7)   # as after a first call
    assert flint_lib.stream_handle(None) == 7
    pid = os.fork()
    if pid == 0:
        os._exit(0 if flint_lib._current_stream is flint_lib._first_current_stream else 1)
    _, status = os.waitpid(pid, 0)
    assert os.waitstatus_to_exitcode(status) == 0
    assert flint_lib.stream_handle(None) == 7   # the parent keeps its own
