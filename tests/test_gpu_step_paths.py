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


def refine_mixed(g):
    """A level-1 tree with its first leaf refined, and in that family the last
    again: faces of all three relations."""
    g.refine_all()
    for leaf in (0, (1 << g.rank) - 1):
        flags = np.zeros(g.size(), dtype=np.int8)
        flags[leaf] = 1
        assert g.reconstruct_tree(flags)


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


def upwind_of_padded(g, vel, dt):
    """One step in numpy from the library's padded patches (the halos that
    brute-force geometry checks elsewhere), in time_step_cpu's expression
    order."""
    pad = g.get_patches()
    level = (g.keys() & np.uint64(63)).astype(np.int64)
    cs = g.cell_sizes(level)
    h, rank = g.halo, g.rank
    core = tuple(slice(h, -h) for _ in range(rank))
    u = pad[(slice(None),) + core]
    total = np.zeros_like(u)
    for d in range(rank):
        j = rank - 1 - d
        lo, hi = list(core), list(core)
        lo[j], hi[j] = slice(h - 1, -h - 1), slice(h + 1, pad.shape[1 + j] - h + 1)
        lo, hi = pad[(slice(None), *lo)], pad[(slice(None), *hi)]
        v, hs = vel[d], 0.5 * abs(vel[d])
        right = 0.5 * (u * v + hi * v) - hs * (hi - u)
        left = 0.5 * (lo * v + u * v) - hs * (u - lo)
        total -= (dt / cs[:, d]).reshape((-1,) + (1,) * rank) * (right - left)
    return u + total


# (rank, extents): one pass and several, partial last pass, a layer as wide as
# the workgroup and wider, more ghost items than threads, the smallest patch,
# and a tile just too large for LDS (memory path)
BOXES = [(2, (2, 2)), (2, (2, 128)), (2, (130, 4)), (2, (6, 300)), (2, (90, 88)), (2, (94, 94)), (3, (2, 2, 2)),
         (3, (12, 10, 6)), (3, (6, 16, 16)), (3, (4, 18, 20)), (3, (16, 16, 16)), (3, (2, 4, 30))]


@pytest.mark.parametrize("rank,ext", BOXES)
def test_any_shape_tiles(amr, rank, ext):
    """Steps of patches that the tile kernel walks in different ways, on a
    tree with same-level, finer and coarser faces."""
    say(f"case: any-shape tile {ext}")
    vel = (1.0, -0.5, 0.25)[:rank]
    g = amr.NdTree(rank, 4, ext, 1, 200)
    s = amr.AmrSolver(g, vel, 0.4)
    refine_mixed(g)
    g.set_interior(np.random.default_rng(sum(ext)).standard_normal(g.size() * g.ni))
    for step in range(3):
        exp = upwind_of_padded(g, vel, s.compute_dt())
        s.advance()
        assert_fields(g.get_interior(), exp, f"{ext} step {step}")


@pytest.mark.parametrize("vel", [(1.0, -0.5, 0.25), (-0.3, 0.0, -1.0)])
@pytest.mark.parametrize("rank,n", [(2, 16), (3, 8)])
def test_adjoint_wave_kernels(amr, rank, n, vel):
    """The one-wave-per-leaf adjoint steps (one ghost layer) against the
    any-shape ones, which serve the same patches with two ghost layers: the
    same sums in the same order, on a tree with same-level, finer and coarser
    faces on every side, and on the root alone."""
    import torch

    say(f"case: adjoint of {n}^{rank} patches, velocity {vel}")
    for adapted in (True, False):
        got = []
        for halo in (1, 2):
            g = amr.NdTree(rank, 4, n, halo, 200)
            s = amr.AmrSolver(g, vel[:rank], 0.4)
            if adapted:
                refine_mixed(g)
            rng = np.random.default_rng(3)
            u0 = rng.standard_normal(g.size() * g.ni)
            g.set_interior(u0)
            tape = amr.Tape(s, 3, None, 0, 2)
            u = torch.from_numpy(u0).cuda()
            lam = torch.from_numpy(rng.standard_normal(u0.size)).cuda()
            uT, grad = torch.empty_like(u), torch.empty_like(u)
            tape.forward(u.data_ptr(), vel[:rank], uT.data_ptr())
            gv = tape.adjoint(lam.data_ptr(), grad.data_ptr())
            got.append((uT.cpu().numpy(), grad.cpu().numpy(), gv))
        for a, b, what in zip(*got, ("uT", "grad_u0", "grad_v")):
            assert np.array_equal(a, b), (adapted, what, np.abs(a - b).max())
