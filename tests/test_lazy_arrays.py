"""Arrays made on their first use (``_kept``): which stream waits for which,
and what a graph capture keeps, with the streams played by numbers."""

from __future__ import annotations

import types

import pytest
import torch


class _Streams:
    """Stands in for the extension: the current stream and capture, the
    streams that are captured elsewhere, and the joins that were made."""

    def __init__(self):
        self.now = (1, 0)
        self.captured = set()
        self.joins = []

    def current_stream(self, device):
        return self.now[0]

    def stream_state(self, device):
        return self.now

    def join_stream(self, device, writer):
        if writer in self.captured:
            return False
        self.joins.append((self.now[0], writer))
        return True


@pytest.fixture
def streams(monkeypatch):
    import mlx_lattice_amd._native as native

    fake = _Streams()
    monkeypatch.setattr(native, 'ext', fake)
    monkeypatch.setattr(torch.cuda, 'current_stream', lambda device: None)
    return fake


def _lazy():
    from mlx_lattice_amd.core.relations.views import _kept

    holder = types.SimpleNamespace(value=None, _written={})
    made = []

    def get():
        def make():
            made.append(object())
            return made[-1]

        return _kept(holder, 'value', torch.device('cuda', 0), make)

    return holder, made, get


def test_another_stream_waits_once(streams):
    holder, made, get = _lazy()
    first = get()
    assert get() is first and holder.value is first and not streams.joins
    streams.now = (2, 0)
    assert get() is first and get() is first
    assert streams.joins == [(2, 1)] and len(made) == 1
    streams.now = (3, 0)
    get()
    assert streams.joins == [(2, 1), (3, 1)]
    # reset, the next use writes on its own stream
    holder.value = None
    second = get()
    assert second is not first and len(made) == 2
    streams.now = (1, 0)
    assert get() is second and streams.joins[-1] == (1, 3)


def test_a_capture_keeps_its_arrays_to_itself(streams):
    holder, made, get = _lazy()
    streams.now = (1, 7)
    first = get()
    assert get() is first and holder.value is None
    streams.now = (1, 8)          # the next graph
    assert get() is not first and holder.value is None
    streams.now = (2, 8)          # a fork of it
    get()
    assert len(made) == 3
    streams.now = (1, 0)          # eager, before any replay
    eager = get()
    assert eager is made[3] and holder.value is eager
    streams.now = (2, 9)          # made before the capture
    assert get() is eager and not streams.joins and len(made) == 4


def test_a_writer_under_capture_is_not_waited_for(streams):
    holder, made, get = _lazy()
    first = get()
    streams.now, streams.captured = (2, 0), {1}
    assert get() is made[1] and holder.value is first
    streams.captured = set()
    assert get() is first and streams.joins == [(2, 1)]


def test_a_given_value_is_nobodys(streams):
    holder, made, get = _lazy()
    holder.value = given = object()
    for state in ((1, 0), (2, 0), (2, 5)):
        streams.now = state
        assert get() is given
    assert not made and not streams.joins
