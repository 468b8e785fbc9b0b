"""Host buffers to and from the device through the pinned staging: every byte comes back, for
sizes below and above the staged path's threshold (2 MB), with a part chunk at the end, with one
and several threads of its own, and from two host threads at once (one of them then takes the
runtime's path)."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def round_trip(gpu, N, seed, times=1):
    ctx = gpu.Context(gpu.make_config(N=N))
    rng = np.random.default_rng(seed)
    for _ in range(times):
        P = rng.normal(size=ctx.shape)
        ctx.upload(P)
        assert np.array_equal(ctx.download(), P)
        a = rng.normal(size=N)
        ctx.upload_field(3, a)
        assert np.array_equal(ctx.download_field(3), a)
    ctx.close()


@pytest.mark.parametrize("N", [(25, 26, 27), (26, 26, 26), (59, 61, 67), (66, 66, 67), (131, 94, 113)])
def test_round_trip(gpu, N):
    round_trip(gpu, N, sum(N))


def test_two_threads(gpu):
    failures = []

    def run(N, seed):
        try:
            round_trip(gpu, N, seed, times=4)
        except BaseException as e:
            failures.append(e)

    threads = [threading.Thread(target=run, args=((80, 70, 64 + k), k)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures
