"""Launches beside the main stream: it waits for them before the caller gives any buffer back, also when one of them raises."""

import contextlib

import pytest
import torch

from primus_amd.pytorch import ops


@pytest.mark.parametrize("raises", [False, True])
def test_the_main_stream_waits(monkeypatch, raises):
    seen = []

    class Stream:
        def wait_stream(self, other):
            seen.append((self, other))

    @contextlib.contextmanager
    def stream(s):
        seen.append(s)
        try:
            yield
        finally:
            seen.append("back")

    monkeypatch.setattr(torch.cuda, "stream", stream)
    main, side = Stream(), Stream()
    with pytest.raises(RuntimeError) if raises else contextlib.nullcontext():
        with ops._beside(main, side):
            seen.append("launch")
            if raises:
                raise RuntimeError
    assert seen == [side, "launch", "back", (main, side)]
