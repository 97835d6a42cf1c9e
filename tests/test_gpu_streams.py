"""Calls whose halves run on different streams, or on streams of different threads, while one of them is busy."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _busy(stream, milliseconds=100):
    """Queues work on ``stream`` that takes about this long or longer; an event behind it."""
    import torch

    x = torch.ones(1 << 28, device="cuda")
    with torch.cuda.stream(stream):
        for _ in range(4 * milliseconds):  # 2 GiB read and written
            x.mul_(1.0)
        done = torch.cuda.Event()
        done.record()
    x.record_stream(stream)
    return done


@pytest.mark.parametrize("granularity", ["inter-stage", "uniform-device-pp", "uniform-pp"])
def test_a_search_built_on_one_stream_runs_on_another(granularity):
    import torch

    from mist_amd.tune_one_case import PreparedSearch
    from tests.util import load_plan

    cfg, _ = load_plan(1, tuning__tuning_granularity=granularity)
    want = PreparedSearch(cfg).run()
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(a):
        PreparedSearch(cfg).run()  # (memory of the stream, so that nothing below waits for some)
    torch.cuda.synchronize()
    done = _busy(a)
    with torch.cuda.stream(a):
        search = PreparedSearch(cfg)
    assert not done.query(), "the upload is not there yet"
    with torch.cuda.stream(b):
        # what a launch does before its kernels
        search.tuner.launch(search.plan, dict(search.dev_plan, batches=[]), None)
        assert not b.query(), "the launch waits for nothing"
        got = search.run()
    assert done.query() and got == want
