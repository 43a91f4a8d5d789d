"""Graph captures run with the cyclic garbage collector held off, and leave it as it was (host, no GPU)."""
import contextlib
import gc

import pytest

from pgj import _chunks


class _Cycle:
    deleted = []

    def __init__(self):
        self.me = self

    def __del__(self):
        _Cycle.deleted.append(gc.isenabled())


@pytest.mark.parametrize('enabled', [True, False])
@pytest.mark.parametrize('fails', [False, True])
def test_no_collection_inside_a_capture(monkeypatch, enabled, fails):
    @contextlib.contextmanager
    def graph(g):
        yield
    monkeypatch.setattr(_chunks.torch.cuda, 'graph', graph)
    was, thresholds = gc.isenabled(), gc.get_threshold()
    try:
        gc.collect()
        (gc.enable if enabled else gc.disable)()
        _Cycle.deleted.clear()
        with contextlib.suppress(RuntimeError):
            with _chunks.capturing(object()):
                gc.set_threshold(1, 1, 1)      # any allocation would start a collection
                _Cycle()
                keep = [[] for _ in range(2000)]
                assert not gc.isenabled() and not _Cycle.deleted and len(keep) == 2000
                if fails:
                    raise RuntimeError('launch failed')
        assert gc.isenabled() is enabled
    finally:
        gc.set_threshold(*thresholds)
        (gc.enable if was else gc.disable)()
        gc.collect()
