"""The batched autotuner's choice of what it times, on the host: the solve that the
whole batch's candidates shape, on a sample that runs in the same kernel."""
import os
import re

import numpy as np

from tnl_amd import batched as B

CSRC = os.path.join(os.path.dirname(os.path.abspath(B.__file__)), "csrc")


def _batch(sizes, wide=()):
    """Diagonal blocks: tridiagonal, rows of 9 slots in the systems `wide`."""
    off, cols, rows = [0], [], [0]
    for k, n in enumerate(sizes):
        for r in range(n):
            c = sorted({max(0, r - 1), r, min(n - 1, r + 1)})
            if k in wide:
                c = list(range(min(n, 9)))
            cols += [rows[-1] + j for j in c]
            off.append(len(cols))
        rows.append(rows[-1] + n)
    cols = np.array(cols, np.int32)
    return np.array(off, np.int32), cols, np.arange(len(cols), dtype=np.float64), np.array(rows, np.int64)


def test_limits_are_the_kernels():
    text = open(os.path.join(CSRC, "batched.hip")).read()
    assert int(re.search(r"kLocalMost = (\d+)", text).group(1)) == B.LOCAL_ROWS
    assert int(re.search(r"kLocalWidth = (\d+)", text).group(1)) == B.LOCAL_SLOTS


def test_whole_batch_decides():
    # (sizes, systems of wide rows, first k) -> (mixed is timed, system added to the sample)
    big = B.LOCAL_ROWS + 1
    for sizes, wide, k, mixed, added in (([5, 7, 6, 9], (), 2, True, None), ([5, 7, 6, big], (), 2, False, 3),
                                         ([5, big, 6, big], (), 2, False, None), ([5, 7, 12, 9], (2,), 2, False, 2),
                                         ([12, 7, 6], (0,), 2, False, None), ([5, 7, 12, big], (2,), 1, False, 2),
                                         ([B.LOCAL_ROWS, 3], (), 1, True, None)):
        off, cols, vals, rows = _batch(sizes, wide)
        o, c, v, s, timed = B._sample(off, cols, vals, rows, k)
        assert timed == mixed
        systems = list(range(k)) + ([added] if added is not None else [])
        assert list(np.diff(s)) == [sizes[j] for j in systems]
        assert len(o) == s[-1] + 1 and o[-1] == len(c) == len(v)
        for at, j in enumerate(systems):  # each sampled system is the batch's, its columns its own
            for r in range(sizes[j]):
                got, want = slice(o[s[at] + r], o[s[at] + r + 1]), slice(off[rows[j] + r], off[rows[j] + r + 1])
                assert np.array_equal(c[got] - s[at], cols[want] - rows[j])
                assert np.array_equal(v[got], vals[want])
