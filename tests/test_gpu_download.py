"""Large results to host memory: sizes around the staged copy's threshold
(8 MiB) and its 1 MiB chunks, pageable and pinned destinations, handles side
by side in several threads."""
import threading

import numpy as np
import pytest
import torch

import vring_amd

pytestmark = pytest.mark.gpu


def roundtrip(s, shape, seed):
    a = np.random.default_rng(seed).standard_normal(shape)
    s.upload("q1", a)
    assert np.array_equal(s.download("q1"), a)
    s.upload("q1", -a)
    assert np.array_equal(s.download("q1"), -a)


# haloed fields of (nt, nr + 3, nz + 3): just below 8 MiB, 8 MiB, a short last
# chunk, 24 whole chunks, one value more than a chunk's multiple in odd sizes
@pytest.mark.parametrize("nt,nr,nz", [(64, 61, 252), (64, 61, 253), (64, 61, 254), (96, 61, 509), (97, 88, 123)])
def test_download_sizes(nt, nr, nz):
    print(f"case download {nt}x{nr}x{nz}", flush=True)
    s = vring_amd.Solver(nt, nr, nz, 4.0, 12.0, 1000.0, 0.01)
    roundtrip(s, (nt, nr + 3, nz + 3), nt)


def test_download_into_pinned_memory():
    nt, nr, nz = 64, 61, 300
    print("case download into pinned memory", flush=True)
    s = vring_amd.Solver(nt, nr, nz, 4.0, 12.0, 1000.0, 0.01)
    a = np.random.default_rng(1).standard_normal((nt, nr + 3, nz + 3))
    s.upload("q1", a)
    pin = torch.zeros(a.size, dtype=torch.float64, pin_memory=True).numpy()
    assert s.L.vrh_download_state(s.h, b"q1", pin) == 0
    assert np.array_equal(pin.reshape(a.shape, order="F"), a)


def test_downloads_of_handles_in_threads():
    nt, nr, nz = 64, 61, 270
    print("case downloads in threads", flush=True)
    hs = [vring_amd.Solver(nt, nr, nz, 4.0, 12.0, 1000.0, 0.01) for _ in range(3)]
    bad = []

    def work(q):
        try:
            for n in range(3):
                roundtrip(hs[q], (nt, nr + 3, nz + 3), 10 * q + n)
        except BaseException as e:
            bad.append(e)

    th = [threading.Thread(target=work, args=(q,)) for q in range(3)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad, bad


def test_downloads_of_one_handle_in_threads():
    nt, nr, nz = 64, 61, 270
    print("case downloads of one handle in threads", flush=True)
    s = vring_amd.Solver(nt, nr, nz, 4.0, 12.0, 1000.0, 0.01)
    want = {n: np.random.default_rng(q).standard_normal((nt, nr + 3, nz + 3)) for q, n in enumerate(("q1", "q2", "q3"))}
    for n, a in want.items():
        s.upload(n, a)
    bad = []

    def work(n):
        try:
            for _ in range(4):
                assert np.array_equal(s.download(n), want[n]), n
        except BaseException as e:
            bad.append(e)

    th = [threading.Thread(target=work, args=(n,)) for n in want]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad, bad


# the same through the pinned slots, which a handle makes once it has fetched 64 MB
@pytest.mark.parametrize("nt,nr,nz", [(64, 61, 253), (64, 61, 254), (96, 61, 509), (97, 88, 123)])
def test_download_sizes_staged(nt, nr, nz):
    print(f"case staged download {nt}x{nr}x{nz}", flush=True)
    s = vring_amd.Solver(nt, nr, nz, 4.0, 12.0, 1000.0, 0.01)
    for _ in range(8):
        s.download("q2")
    roundtrip(s, (nt, nr + 3, nz + 3), nt)
