"""Which taps of the deskew need the row's first/last range: output cell (i, j)
of a sector reads the skewed rows t_j + i and t_j + i + 1, i.e. rows t_j + e
with 0 <= e <= n.  The GPU deskew reads every tap with 0 < e < n unseen and
looks at first/last for e = 0 and e = n only; here the maps of every sector are
checked to allow that, on small sides where each can differ and on large ones
where a table that steps differently once would show."""
import numpy as np
import pytest

import skewengine_amd as ske


@pytest.mark.parametrize("sides", [range(2, 70), (97, 128, 250, 251), (500, 512, 750), (1000, 1024, 1501), (2047,),
                                   (4600,)])
def test_inner_taps_lie_in_their_rows_range(sides):
    for n in sides:
        j = np.arange(n)
        for a in range(180):
            p, t, _, first, last = ske.plan_sector(n, n, a)
            t = t[:n].astype(np.int64)
            assert t[0] >= 0 and np.isin(np.diff(t), (0, 1)).all(), (n, a)
            # rows t_j .. t_j + n - 1 exist
            assert t[-1] + n - 1 < p.skewHeight, (n, a)
            # e = 0: never left of the row's first cell; e = n: inside its row where that row exists
            assert (first[t] <= j).all(), (n, a)
            e = t + n
            assert p.newAngle == 0 or (e < p.skewHeight).all(), (n, a)
            e, je = e[e < p.skewHeight], j[e < p.skewHeight]
            assert ((first[e] <= je) & (je < last[e])).all(), (n, a)
            # column j is inside every row of [t_j + 1, t_j + n - 1] if the rows that exclude it,
            # found from both tables, lie outside that span
            assert (first[:p.skewHeight] <= last[:p.skewHeight]).all()
            for r in range(p.skewHeight):
                lo, hi = int(first[r]), int(last[r])
                # t is nondecreasing: columns with t_j + 1 <= r <= t_j + n - 1 form one span
                c0 = int(np.searchsorted(t, r - n + 1, "left"))
                c1 = int(np.searchsorted(t, r - 1, "right"))
                if c0 < c1:
                    assert lo <= c0 and c1 <= hi, (n, a, r)
