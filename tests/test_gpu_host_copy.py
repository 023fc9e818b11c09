"""Whole arrays between the caller's memory and the device: below the size from which the copy is cut into pinned
chunks, at it, and with a ragged last chunk; from several threads at once, on contexts of their own and on one.

The copies carry bytes: a state that was handed over comes back bit for bit. Its spectrum is numpy's within 1e-12
of the largest mode (eps log2 N with a wide margin)."""
import threading

import numpy as np
import pytest

from tests.helpers import params

pytestmark = pytest.mark.gpu


def _state(n, seed):
    rng = np.random.default_rng(seed)
    uu = 1.0 + 0.1 * rng.standard_normal((8,) + n[::-1]).T
    pr = 1.0 + 0.1 * rng.standard_normal((4,) + n[::-1]).T
    return np.asfortranarray(uu), np.asfortranarray(pr)


# conserved / primitive arrays of 2/1, 8/4, 9/4.5, 12/6 and 48/24 MB
@pytest.mark.parametrize("n", ((32, 32, 32), (64, 64, 32), (96, 96, 16), (96, 64, 32), (128, 96, 64)))
def test_round_trip(n):
    from laps_amd.runtime import Laps
    uu, pr = _state(n, sum(n))
    with Laps(params(n)) as g:
        g.set_state(uu, pr)
        for _ in range(2):
            a, b = g.state()
            assert np.array_equal(a, uu) and np.array_equal(b, pr)
        s = g.spectral()
        for f in (0, 7):
            ref = np.fft.rfftn(uu[..., f].T).T / np.prod(n)
            assert np.abs(s[..., f] - ref).max() <= 1e-12 * np.abs(ref).max()


def test_threads():
    from laps_amd.runtime import Laps
    n = (96, 64, 32)
    states = [_state(n, i) for i in range(3)]
    boxes = [Laps(params(n)) for _ in states]
    wrong = []

    def work(i, g, own):
        for _ in range(3):
            if own:
                g.set_state(*states[i])
            a, b = g.state()
            if not (np.array_equal(a, states[i][0]) and np.array_equal(b, states[i][1])):
                wrong.append(i)

    for own in (True, False):
        th = [threading.Thread(target=work, args=(i if own else 1, boxes[i if own else 1], own)) for i in range(3)]
        for t in th:
            t.start()
        for t in th:
            t.join()
    for g in boxes:
        g.close()
    assert not wrong
