"""The server's collection window, without a GPU: a mini-batch waits for
more requests of its kind while another worker solves, and only then.
Workers that are themselves waiting do not keep each other waiting."""
import threading
import time

import pytest

from tahoe_amd import api, rve, serve

LINGER = 3.0      # s: far above what starting an idle worker takes


def request(rid, L):
    return rve.Request(rid, L, api.TOTAL_LAGRANGIAN, 0.3, seed=5 + rid)


class Clock(serve.RVEServer):
    """Solves nothing: notes when a mini-batch would start, and holds the
    ones of edge 4 until `release`."""

    def __init__(self, **kw):
        super().__init__(workers=3, linger=LINGER, **kw)
        self.started = {}
        self.release = threading.Event()

    def _solve(self, bid, reqs, t0):
        now = time.perf_counter()
        for r in reqs:
            self.started[r.rid] = (now, bid)
        if reqs[0].L == 4:
            assert self.release.wait(30.0)
        return [serve.Result(r.rid, None, 0, r.arrival, 0.0, 0.0, bid, len(reqs)) for r in reqs]

    def put(self, *reqs):
        with self._lock:
            self._queue.extend(reqs)
            self._lock.notify_all()

    def wait_for(self, rid, timeout):
        end = time.perf_counter() + timeout
        while rid not in self.started and time.perf_counter() < end:
            time.sleep(0.002)
        return rid in self.started


@pytest.fixture
def server():
    s = Clock()
    threads = [threading.Thread(target=s._worker, args=(0.0,), daemon=True) for _ in range(3)]
    for t in threads:
        t.start()
    yield s
    s.release.set()
    with s._lock:
        s._closed = True
        s._lock.notify_all()
    for t in threads:
        t.join(30.0)
        assert not t.is_alive()


def test_waiting_workers_do_not_hold_each_other(server):
    server.put(request(0, 4))
    assert server.wait_for(0, 2.0)                      # an idle server starts at once
    server.put(request(1, 10), request(2, 18))          # two more size classes: both workers wait
    time.sleep(0.3)
    assert 1 not in server.started and 2 not in server.started
    server.put(request(3, 10))                          # joins the batch that waits
    time.sleep(0.1)
    t = time.perf_counter()
    server.release.set()                                # nobody solves any more
    assert server.wait_for(1, 10.0) and server.wait_for(2, 10.0) and server.wait_for(3, 10.0)
    assert max(server.started[k][0] for k in (1, 2, 3)) - t < 0.5 * LINGER
    assert server.started[1][1] == server.started[3][1] != server.started[2][1]


def test_window_ends_while_another_solves(server):
    server.put(request(0, 4))
    assert server.wait_for(0, 2.0)
    t = time.perf_counter()
    server.put(request(1, 10))
    assert server.wait_for(1, 10.0)
    assert 0.9 * LINGER < server.started[1][0] - t < 3.0 * LINGER


def test_full_batch_does_not_wait():
    s = Clock(max_batch=2)
    s._solving = 1                                       # another worker solves
    s._queue.extend([request(1, 10), request(2, 11), request(3, 12)])
    t = time.perf_counter()
    with s._lock:
        _, reqs, size = s._take_batch()
    assert time.perf_counter() - t < 0.5 * LINGER
    assert [r.rid for r in reqs] == [1, 2] and [r.rid for r in s._queue] == [3]
    assert size == sum(serve.footprint_bytes(r, s.precision) for r in reqs) == s._in_use
