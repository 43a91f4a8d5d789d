"""Captures of several threads that overlap: the collector stays off until the last one has closed (host, no GPU)."""
import contextlib
import gc
import threading

import pytest

from pgj import _chunks


@pytest.fixture
def fake_graph(monkeypatch):
    @contextlib.contextmanager
    def graph(g):
        yield
    monkeypatch.setattr(_chunks.torch.cuda, 'graph', graph)
    was = gc.isenabled()
    yield
    (gc.enable if was else gc.disable)()


@pytest.mark.parametrize('enabled', [True, False])
def test_first_to_leave_keeps_the_collector_off(fake_graph, enabled):
    (gc.enable if enabled else gc.disable)()
    inside, leave = threading.Event(), threading.Event()

    def first():
        with _chunks.capturing(object()):
            inside.set()
            assert leave.wait(30)

    t = threading.Thread(target=first)
    t.start()
    assert inside.wait(30)
    with _chunks.capturing(object()):
        leave.set()
        t.join(30)
        assert not t.is_alive() and not gc.isenabled()
    assert gc.isenabled() is enabled
