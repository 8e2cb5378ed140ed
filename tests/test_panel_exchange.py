"""The order of the LU panel's exchange between workgroups, checked on the CPU:
every interleaving of the workgroups' steps, with the number of record buffers
that lu.hip declares.  A record must never be overwritten while a workgroup
still waits for it, and no workgroup may wait for ever."""
import itertools
import os
import re

import pytest

SOURCE = open(os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "linear-massiv_amd", "csrc",
                           "lu.hip")).read()


def buffers(record):
    """The declared number of buffers of a record array of PanelSync."""
    size = re.search(r"unsigned long long %s\[(\w+)\]\[MAXP\]" % record, SOURCE).group(1)
    if not size.isdigit():
        size = re.search(r"constexpr int %s = (\d+);" % size, SOURCE).group(1)
    return int(size)


def hazard(keys, rows, winners, P):
    """The first overwritten record or standstill of P workgroups over the
    columns whose pivots `winners` own, or None.

    A workgroup's column j, between its barriers:
      1 to 2: its row waves publish key j; its fifth wave receives row j - 1
              from that column's winner
      2 to 3: its row waves store row j; its fifth wave receives all keys j
    A workgroup is (intervals passed, row waves' step done, fifth wave's step
    done); the records' tags follow from these."""
    K = len(winners)

    def written(w, key, buf, count):
        """The last column whose key (or row) w wrote to buffer `buf`; None:
        none yet."""
        t, a, _ = w
        done = (t + a + key) // 2  # the keys (rows) of its first `done` columns are out
        return next((j for j in range(min(done, K) - 1, -1, -1) if j % count == buf), None)

    def waits(w):
        """(key or row, column, workgroups) that w's fifth wave waits for."""
        j, second = divmod(w[0], 2)
        if second:
            return 1, j, range(P)
        return (0, j - 1, [winners[j - 1]]) if j > 0 else None

    start = ((0, 0, 0),) * P
    seen, todo = {start}, [start]
    while todo:
        state = todo.pop()
        after = []
        for i, w in enumerate(state):
            t, a, b = w
            if t > 2 * K:
                continue
            last = t == 2 * K  # after the columns: only the last row is received
            if not a and not last:
                after.append((i, (t, 1, b)))
            if not b:
                want, ready = waits(w), True
                if want:
                    key, j, whom = want
                    count = keys if key else rows
                    for v in whom:
                        tag = written(state[v], key, j % count, count)
                        if tag is not None and tag > j:
                            return f"{'key' if key else 'row'} {j} of workgroup {v} gone before {i} had it"
                        ready = ready and tag == j
                if ready:
                    after.append((i, (t, a, 1)))
            if (a or last) and b:
                after.append((i, (t + 1, 0, 0)))
        if not after and any(w[0] <= 2 * K for w in state):
            return f"standstill at {state}"
        for i, w in after:
            nxt = state[:i] + (w,) + state[i + 1:]
            if nxt not in seen:
                seen.add(nxt)
                todo.append(nxt)
    return None


@pytest.mark.parametrize("P,K", [(2, 7), (3, 5)])
def test_no_record_is_overwritten_before_it_is_read(P, K):
    for winners in itertools.product(range(P), repeat=K):
        assert hazard(buffers("key"), buffers("row"), winners, P) is None


def test_the_model_finds_too_few_buffers():
    every = list(itertools.product(range(2), repeat=5))
    assert any(hazard(2, 2, w, 2) for w in every)
    assert any(hazard(1, 3, w, 2) for w in every)


def test_row_records_are_indexed_by_their_slot():
    uses = re.findall(r"sy->row\[(\w+)", SOURCE)
    assert uses and all(u == "row_slot" for u in uses)
