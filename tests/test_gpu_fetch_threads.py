"""Tables fetched by several threads, each on a stream of its own."""
import threading

import numpy as np
import pytest

from tests.test_gpu_streams import _busy

pytestmark = pytest.mark.gpu


def _fetch_on(stream, source):
    import torch

    from mist_amd.intra_tuning import fetch_doubles

    out = np.empty(source.numel(), dtype=np.float64)
    with torch.cuda.stream(stream):
        fetch_doubles(source, out)
    return out


def _free_beside(done, streams):
    """A stream whose kernels run beside those in front of ``done`` (streams share a few hardware queues)."""
    import torch

    passed = []
    for stream in streams:
        with torch.cuda.stream(stream):
            torch.zeros(1, device="cuda").add_(1)
            passed.append(stream.record_event())
    while not done.query():
        for stream, event in zip(streams, passed):
            if event.query():
                return stream
    pytest.skip("no other hardware queue")


def test_a_fetch_does_not_wait_for_another_threads_kernels():
    import torch

    busy, *others = [torch.cuda.Stream() for _ in range(5)]
    sources = [torch.rand(200000, dtype=torch.float64, device="cuda") for _ in range(2)]
    want = [source.cpu().numpy() for source in sources]
    for stream in (busy, *others):  # (whatever is made once)
        assert np.array_equal(_fetch_on(stream, sources[0]), want[0])
    done, found = _busy(busy), []
    free = _free_beside(done, others)
    begun = threading.Event()

    def behind():
        begun.set()
        found.append(_fetch_on(busy, sources[0]))

    thread = threading.Thread(target=behind)
    thread.start()
    begun.wait()
    thread.join(0.01)
    assert np.array_equal(_fetch_on(free, sources[1]), want[1])
    assert not done.query()
    thread.join()
    assert done.query() and np.array_equal(found[0], want[0])


def test_more_threads_than_are_kept_chunks_for():
    import torch

    n_threads, rounds = 9, 20
    sources = [torch.rand(150000 + 1000 * i, dtype=torch.float64, device="cuda") for i in range(n_threads)]
    want = [source.cpu().numpy() for source in sources]
    right = [0] * n_threads

    def fetch(i):
        stream = torch.cuda.Stream()
        for _ in range(rounds):
            right[i] += np.array_equal(_fetch_on(stream, sources[i]), want[i])

    threads = [threading.Thread(target=fetch, args=(i,)) for i in range(n_threads)]
    for thread in threads:
        thread.start()
    for thread in threads:
        thread.join()
    assert right == [rounds] * n_threads
