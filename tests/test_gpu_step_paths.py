"""Step paths chosen by batch length, patch shape and tree size, against the
CPU oracle, bit for bit (neither side contracts, so the tolerance is none)."""
import sys

import numpy as np
import pytest

from amrlib import load_package
from test_gpu_euler import init_both, pair as euler_pair, pulse
from test_gpu_parity import assert_fields

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def amr():
    return load_package()


def test_euler_batch_lengths(amr):
    """Batches of 0 to 7 steps one after another (the dt slots of a batch are
    used in turn), a dt query between the queued steps and their read-back,
    and batches whose time runs out within and before them."""
    say("case: Euler batch lengths")
    s, o = euler_pair(amr, 2, 16, 7, 72)
    for _ in range(2):
        s.tree.refine_all()
        o.refine_all()
    init_both(s, o, pulse(2, (1.0, 1.0), amp=2.0))
    for steps in (1, 1, 2, 0, 3, 4, 5, 1, 6, 7, 2):
        s.advance_batch_async(steps)
        exp = o.advance_batch(steps)
        assert s.compute_dt() == o.compute_dt(), steps
        assert s.finish_advance_batch() == exp, steps
    for steps, share in ((5, 2.5), (4, 1.5), (3, 0.0), (1, 0.5), (4, 10.0)):
        left = share * o.compute_dt()
        s.advance_batch_async(steps, left)
        assert s.finish_advance_batch() == o.advance_batch(steps, left), (steps, share)
    assert_fields(s.tree.get_interior(), o.get_interior(), "after the batches")
