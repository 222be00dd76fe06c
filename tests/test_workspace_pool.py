"""The pools of workspaces (host side): threads that take, evict and release at once."""
import threading
import time

from nha_amd import ops


class _Slow(dict):
    """A dictionary that gives other threads their turn between a key's choice and its removal."""

    def pop(self, *a):
        time.sleep(1e-4)
        return super().pop(*a)


def test_threads_take_evict_and_release_at_once(monkeypatch):
    monkeypatch.setattr(ops, "_WORKSPACE", _Slow())
    monkeypatch.setattr(ops, "_WORKSPACE_MAX_STREAMS", 3)
    failed, held = [], []

    def take(first):
        try:
            for i in range(60):
                ws = ops._workspace(1 << 20, "cpu", first + i % 5)
                assert ws.numel() >= 1 << 20
                if i % 20 == 19:
                    held.append(ops.release_workspaces())
        except Exception as e:
            failed.append(repr(e))
    threads = [threading.Thread(target=take, args=(10 * t,)) for t in range(6)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not failed and len(ops._WORKSPACE) <= 3 and any(held)
