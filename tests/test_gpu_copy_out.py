"""Copies of large objects to pageable memory, which go through pinned slots
and several threads: below and at the smallest such size, with a ragged last
chunk, past the slots, and from two contexts in two threads.  Exact.
"""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _round_trip(rows, seed, out):
    from phasecon_amd.mbir import Stage
    from phasecon_amd.synth import geometry_scan
    st = Stage(geometry_scan(rows, 256, 4))
    x = np.random.default_rng(seed).random(st.shape_x, np.float32)
    for _ in range(3):
        st.set_object(x)
        out.append(np.array_equal(st.get_object(), x))
        x += 1
    st.close()


# 256 KiB per row: 8 MiB less a row, 8 MiB, a ragged chunk, 16 MiB (the
# slots) and a row, 33 MiB less a row
@pytest.mark.parametrize("rows", [31, 32, 33, 65, 131])
def test_large_copies_are_exact(rows):
    out = []
    _round_trip(rows, rows, out)
    assert out == [True] * 3


def test_two_contexts_in_two_threads():
    out = [[], []]
    th = [threading.Thread(target=_round_trip, args=(65 + i, i, out[i])) for i in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert out == [[True] * 3] * 2
