"""The threads that help with large host arrays (tq_host_serve), with the test in the driver's place: no GPU needed."""
import ctypes as C
import threading
import time

import numpy as np
import pytest

from turboquant_plus_amd import _lib as L


class Job:
    """A fetch of n_pieces pieces whose slots are filled already; the test lets pieces be worked on."""

    def __init__(self, n_pieces, piece=4096, kind=L.HOST_FETCH):
        assert n_pieces <= L.HOST_SLOTS
        n = n_pieces * piece - 7
        self.slots = np.random.default_rng(n).integers(0, 256, n_pieces * piece).astype(np.uint8)
        self.host = np.zeros(n, np.uint8)
        self.job = L.TQHostJob(kind=kind, n=n, n_pieces=n_pieces, piece=piece, host=self.host.ctypes.data, slots=self.slots.ctypes.data)

    def post(self, board, at):
        board.desk[at].taken = 1
        board.desk[at].job = C.addressof(self.job)
        wake(board)

    def allow(self, board, upto):
        self.job.ready = upto
        wake(board)

    def wait(self, done, seconds=20):
        end = time.time() + seconds
        while self.job.done < done and time.time() < end:
            time.sleep(0.001)
        return self.job.done == done

    def take_away(self, board, at):
        board.desk[at].job = None
        while board.desk[at].users:
            time.sleep(0.001)
        board.desk[at].taken = 0


def wake(board):
    L.lib().tq_host_open(board, 0)
    L.lib().tq_host_close(board, 0)


def users(board):
    return board.state >> 32


def serving(board):
    return board.state & 0xFFFFFFFF


def serve(board, count):
    assert L.lib().tq_host_open(board, count) == count
    threads = [threading.Thread(target=L.lib().tq_host_serve, args=(board,)) for _ in range(count)]
    for t in threads:
        t.start()
    return threads


def close(board, threads):
    L.lib().tq_host_close(board, 0)
    for t in threads:
        t.join(20)
        assert not t.is_alive()
    assert board.state == 0


def test_waiting_costs_no_processor_time():
    """A job whose pieces are not there yet (the stream has other work before them) and a board without jobs."""
    board, job = L.TQHostBoard(), Job(4)
    threads = serve(board, 6)
    for post in (False, True):
        if post:
            job.post(board, 0)
        time.sleep(0.05)
        before = time.process_time()
        time.sleep(0.6)
        assert time.process_time() - before < 0.15      # six threads that spin take 3.6 s where there are as many processors
    for k in (1, 2, 4):
        job.allow(board, k)
        assert job.wait(k)
    assert np.array_equal(job.host, job.slots[:job.host.size])
    job.take_away(board, 0)
    close(board, threads)


@pytest.mark.parametrize("count", [1, 3])
def test_a_job_that_waits_keeps_nobody_from_another(count):
    board, stuck, other = L.TQHostBoard(), Job(3), Job(8)
    stuck.post(board, 2)
    threads = serve(board, count)
    time.sleep(0.05)
    other.post(board, 5)
    other.allow(board, 8)
    assert other.wait(8) and stuck.job.done == 0
    other.take_away(board, 5)
    stuck.allow(board, 3)
    assert stuck.wait(3)
    stuck.take_away(board, 2)
    close(board, threads)
    for j in (stuck, other):
        assert np.array_equal(j.host, j.slots[:j.host.size])


def back_in_the_pool():
    together = threading.Barrier(L.COPY_THREADS + 1)
    for _ in range(L.COPY_THREADS):
        L._copy_pool().submit(together.wait)
    together.wait(20)
    return L._board.state == 0


def test_two_callers_share_the_copy_threads():
    """A caller that only waits for its device work has the threads to itself no longer than another one has an array under way."""
    inside, leave = threading.Event(), threading.Event()

    def first():
        with L.helpers(L.SHARED + 1):
            inside.set()
            leave.wait(30)
    t = threading.Thread(target=first)
    t.start()
    assert inside.wait(20)
    job = Job(8)
    queued = L._copy_pool()._work_queue.qsize()
    with L.helpers(L.SHARED + 1):
        job.post(L._board, 0)
        job.allow(L._board, 8)
        assert job.wait(8)
        job.take_away(L._board, 0)
        assert L._copy_pool()._work_queue.qsize() <= queued      # nothing is left there for threads that are busy
    leave.set()
    t.join(20)
    assert np.array_equal(job.host, job.slots[:job.host.size]) and back_in_the_pool()
    with L.helpers(L.SHARED + 1):
        job2 = Job(2)
        job2.post(L._board, 1)
        job2.allow(L._board, 2)
        assert job2.wait(2)
        job2.take_away(L._board, 1)
    assert back_in_the_pool()


def test_threads_that_cannot_be_had(monkeypatch):
    """The count of threads at the board holds where a submit fails, also one that has queued its work; without threads, too."""
    pool, sent = L._copy_pool(), []

    class Ending:
        def submit(self, fn, *args):
            pool.submit(fn, *args)
            sent.append(1)
            if len(sent) == 2:
                raise RuntimeError("can't start new thread")
    monkeypatch.setattr(L, "_copy_pool", Ending)
    monkeypatch.setattr(L, "COPY_THREADS", 4)
    with L.helpers(L.SHARED + 1):
        assert len(sent) == 2 and users(L._board) == 1 and serving(L._board) == 4
    assert serving(L._board) <= 2 and users(L._board) == 0
    monkeypatch.undo()
    assert back_in_the_pool()


def test_a_second_call_finds_the_threads_still_there():
    """They leave some milliseconds after the last call, so that calls in a row do not send for them each time."""
    with L.helpers(L.SHARED + 1):
        pass
    assert serving(L._board) == L.COPY_THREADS
    before = L._copy_pool()._work_queue.qsize()
    with L.helpers(L.SHARED + 1):
        assert serving(L._board) == L.COPY_THREADS and L._copy_pool()._work_queue.qsize() <= before
    assert back_in_the_pool()


def test_no_more_threads_than_processors():
    import os
    assert 1 <= L.COPY_THREADS <= max(1, len(os.sched_getaffinity(0)) - 1)
