"""The split of a batch's trees into groups that are stepped one after another:
every group keeps to the limit unless it is one tree larger than that, no split
needs fewer groups, and none of as many has a smaller largest group."""
import numpy as np
import pytest

import emulation as emu


def best_split(sizes, most):
    """(groups, largest group) by dynamic programming over the last group."""
    best = [(0, 0)]
    for end in range(1, len(sizes) + 1):
        options = []
        for start in range(end):
            size = sum(sizes[start:end])
            if size > most and end - start > 1:
                continue
            groups, largest = best[start]
            # a tree above the limit is alone whatever the split: it does not count
            options.append((groups + 1, max(largest, size if size <= most else 0)))
        best.append(min(options))
    return best[-1]


CASES = [([140, 140, 140], 224), ([149, 149, 149], 224), ([150, 230, 60], 224), ([150, 148, 150], 224),
         ([1], 224), ([224], 224), ([225], 224), ([112, 112, 112, 112], 224), ([300, 1, 300, 1, 1], 224),
         ([1] * 500, 224), ([223, 1, 223, 1, 1], 224), ([5, 5, 5], 1)]
RNG = np.random.default_rng(4)
CASES += [(RNG.integers(1, top, RNG.integers(1, 40)).tolist(), 224) for top in (20, 120, 224, 320) for _ in range(20)]


@pytest.mark.parametrize("sizes,most", CASES, ids=lambda v: str(v)[:24])
def test_groups_keep_to_the_limit(sizes, most):
    first = emu.batch_groups(sizes, most)
    assert first[0] == 0 and all(a < b for a, b in zip(first, first[1:])) and first[-1] < len(sizes)
    groups = [sizes[a:b] for a, b in zip(first, first[1:] + [len(sizes)])]
    for g in groups:
        assert sum(g) <= most or len(g) == 1, g
    count, largest = best_split(sizes, most)
    assert len(groups) == count
    assert max([sum(g) for g in groups if sum(g) <= most], default=0) == largest
