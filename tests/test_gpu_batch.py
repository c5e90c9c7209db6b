"""Batched form: many independent trees stepped as one launch (and as one
hipGraph launch) must reproduce the per-tree plain solves and the oracle bit
for bit, with each instance's own velocity and dt."""
import sys

import numpy as np
import pytest

from amrlib import load_package
from oracle import OracleTree

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def amr():
    mod = load_package()
    import gpu_amr_amd.workloads  # noqa: F401

    return mod


def build(amr, count, rounds=3, max_depth=6):
    from gpu_amr_amd import workloads

    out = [workloads.c4_instance(amr, i, max_depth=max_depth, rounds=rounds, capacity=4096 + 64) for i in range(count)]
    return out


def test_batch_matches_sequential_and_oracle(amr):
    say("case: batch of 6 C4-style instances, 20 steps, eager launches")
    built = build(amr, 6)
    trees = [b[0] for b in built]
    solvers = [b[1] for b in built]
    init = [t.get_interior().copy() for t in trees]
    batch = amr.Batch(trees)
    assert batch.size() == sum(t.size() for t in trees)
    batch.advance(20, use_graph=False)
    batch.synchronize()
    for s in solvers:
        s.advance_batch_async(20)
        s.finish_advance_batch()
    seq = [t.get_interior().copy() for t in trees]
    batch.scatter()
    for i, (t, u) in enumerate(zip(trees, seq)):
        assert np.array_equal(t.get_interior().view(np.uint64), u.view(np.uint64)), f"instance {i}"
    # the oracle on two instances (replaying the same regrid flags)
    for i in (0, 3):
        _, _, history, vel, _ = built[i]
        o = OracleTree(2, 16, 1, 7, 8192 + 64)
        o.set_params(vel, 0.4, threads=8)
        for _ in range(3):
            o.refine_all()
        for f in history:
            o.reconstruct(f)
        np.testing.assert_array_equal(o.keys(), trees[i].keys())
        o.set_interior(init[i])
        o.halo_exchange()
        o.advance_batch(20)
        assert np.array_equal(o.get_interior().view(np.uint64), seq[i].view(np.uint64)), f"oracle instance {i} v={vel}"


def test_batch_graph_replays(amr):
    say("case: batch hipGraph replays vs eager")
    built = build(amr, 4)
    trees = [b[0] for b in built]
    g_batch = amr.Batch(trees)
    e_batch = amr.Batch(trees)
    for rep in range(4):
        g_batch.advance(5, use_graph=True)
        g_batch.synchronize()
        e_batch.advance(5, use_graph=False)
        e_batch.synchronize()
        _ = trees[0].get_interior()  # unrelated eager work between replays
        e_batch.scatter()
        e_res = [t.get_interior().copy() for t in trees]
        g_batch.scatter()
        for i, t in enumerate(trees):
            assert np.array_equal(t.get_interior().view(np.uint64), e_res[i].view(np.uint64)), f"replay {rep} instance {i}"


def test_batch_variants_and_autotune(amr):
    say("case: batch variants")
    built = build(amr, 3)
    trees = [b[0] for b in built]
    ref = amr.Batch(trees)
    ref.advance(4, use_graph=False)
    ref.scatter()
    exp = [t.get_interior().copy() for t in trees]
    ref.close()
    nvar = len(built[0][1].step_variants())
    for v in range(nvar):
        # rebuild from the same initial state each time
        fresh = build(amr, 3)
        tr = [b[0] for b in fresh]
        bt = amr.Batch(tr)
        bt.set_step_variant(v)
        bt.advance(4, use_graph=(v % 2 == 0))
        bt.scatter()
        for i, t in enumerate(tr):
            assert np.array_equal(t.get_interior().view(np.uint64), exp[i].view(np.uint64)), f"variant {v} instance {i}"
    best, us = bt.autotune(3)
    assert 0 <= best < nvar and us > 0


def test_batch_run_variant_with_graphs_and_switches(amr):
    say("case: batch run8 graph replays with variant switches")
    built = build(amr, 4)
    trees = [b[0] for b in built]
    names = built[0][1].step_variants()
    rv = names.index("run8")
    ref = amr.Batch(trees)
    bt = amr.Batch(trees)
    plan = [(rv, True, 4), (0, True, 3), (rv, True, 4), (rv, False, 1), (1, False, 2), (rv, True, 4), (rv, True, 3)]
    for i, (v, graph, steps) in enumerate(plan):
        bt.set_step_variant(v)
        bt.advance(steps, use_graph=graph)
        bt.synchronize()
        ref.advance(steps, use_graph=False)
        ref.synchronize()
        ref.scatter()
        exp = [t.get_interior().copy() for t in trees]
        bt.scatter()
        for k, t in enumerate(trees):
            assert np.array_equal(t.get_interior().view(np.uint64), exp[k].view(np.uint64)), f"plan step {i} instance {k}"


@pytest.mark.parametrize("rank,n,level", [(2, 16, 7), (3, 8, 5), (2, 64, 5)])
def test_batch_larger_than_the_cache_matches_sequential(amr, rank, n, level):
    """A batch that is stepped in several groups of instances: uneven trees,
    odd and even step counts, eager and graph launches, per-leaf and run
    kernels."""
    say(f"case: batch of {n}^{rank} patches in several groups")
    cells = n**rank
    solvers = []
    leaves = 0
    rng = np.random.default_rng(level)
    while leaves * cells * 16 < 460e6:  # groups hold at most 224 MiB
        k = level if len(solvers) % 3 else level - 1
        tree = amr.NdTree(rank, level, n, 1, (1 << (rank * k)) + 1)
        solvers.append(amr.AmrSolver(tree, tuple(rng.uniform(-1.0, 1.0, rank)), 0.4))
        for _ in range(k):
            tree.refine_all()
        tree.set_interior(rng.standard_normal(tree.size() * tree.ni))
        leaves += tree.size()
    batch = amr.Batch([s.tree for s in solvers])
    steps = 0
    for variant, count, graph in ((0, 3, True), (4 if n < 64 else 0, 2, False), (0, 1, False), (0, 3, True)):
        batch.set_step_variant(variant)
        batch.advance(count, use_graph=graph)
        steps += count
    batch.synchronize()
    expected = []
    for s in solvers:
        s.advance_batch_async(steps)
        s.finish_advance_batch()
        expected.append(s.tree.get_interior().copy())
    batch.scatter()
    for i, (s, u) in enumerate(zip(solvers, expected)):
        assert np.array_equal(s.tree.get_interior().view(np.uint64), u.view(np.uint64)), f"instance {i}"


def test_batch_of_groups_short_and_long_calls(amr):
    """Calls of one to four steps on a batch of several groups (the short ones
    run on all leaves at once), per-leaf and run kernels, eager and by graph,
    against the sequential solves after every call."""
    say("case: short and long calls on a batch of several groups")
    rng = np.random.default_rng(12)
    solvers = []
    for _ in range(8):  # 8 x 64 MiB of state
        tree = amr.NdTree(2, 7, 16, 1, 1 << 14)
        solvers.append(amr.AmrSolver(tree, tuple(rng.uniform(-1.0, 1.0, 2)), 0.4))
        for _ in range(7):
            tree.refine_all()
        tree.set_interior(rng.standard_normal(tree.size() * tree.ni))
    other = []
    for s in solvers:
        tree = amr.NdTree(2, 7, 16, 1, 1 << 14)
        other.append(amr.AmrSolver(tree, s.velocity, 0.4))
        for _ in range(7):
            tree.refine_all()
        tree.set_interior(s.tree.get_interior())
    batch = amr.Batch([s.tree for s in solvers])
    run8 = solvers[0].step_variants().index("run8")
    for variant, steps, graph in ((0, 1, False), (run8, 3, False), (run8, 1, True), (run8, 1, True), (0, 2, True),
                                  (0, 4, False), (run8, 2, False), (0, 1, True), (0, 1, True), (0, 2, True)):
        batch.set_step_variant(variant)
        batch.advance(steps, use_graph=graph)
        batch.scatter()
        for i, (s, o) in enumerate(zip(solvers, other)):
            o.advance_batch_async(steps)
            o.finish_advance_batch()
            a, b = s.tree.get_interior(), o.tree.get_interior()
            assert np.array_equal(a.view(np.uint64), b.view(np.uint64)), (variant, steps, graph, i)


def test_scatter_refuses_a_regridded_tree(amr):
    """A tree refined or coarsened since the batch was made, first, in the
    middle or last: scatter raises and no tree is written."""
    say("case: scatter into regridded trees")
    for which, flag in ((1, "REFINE"), (1, "COARSEN"), (0, "REFINE"), (2, "REFINE"), (2, "COARSEN")):
        trees = []
        for k in range(3):
            t = amr.NdTree(2, 6, 16, 1, 200)
            s = amr.AmrSolver(t, (1.0, 0.5), 0.4)
            for _ in range(3):
                t.refine_all()
            t.set_interior(np.random.default_rng(k).standard_normal(t.size() * t.ni))
            trees.append((t, s))
        batch = amr.Batch([t for t, _ in trees])
        batch.advance(2, use_graph=False)
        flags = np.zeros(64, dtype=np.int8)
        flags[:4] = getattr(amr, flag)
        assert trees[which][0].reconstruct_tree(flags)
        before = [t.get_interior() for t, _ in trees]
        with pytest.raises(amr.AmrError):
            batch.scatter()
        batch.synchronize()
        for (t, _), u in zip(trees, before):
            assert np.array_equal(t.get_interior().view(np.uint64), u.view(np.uint64)), (which, flag)


def test_batch_of_more_trees_than_a_scatter_launch(amr):
    """300 trees of different sizes: the scatter takes several launches."""
    say("case: batch of 300 trees")
    rng = np.random.default_rng(5)
    solvers, other = [], []
    for k in range(300):
        u = None
        v = tuple(rng.uniform(-1.0, 1.0, 2))
        for made in (solvers, other):
            t = amr.NdTree(2, 4, 8, 1, 16)
            made.append(amr.AmrSolver(t, v, 0.4))
            for _ in range(k % 3):
                t.refine_all()
            u = rng.standard_normal(t.size() * t.ni) if u is None else u
            t.set_interior(u)
    batch = amr.Batch([s.tree for s in solvers])
    batch.advance(3)
    batch.scatter()
    for k, (s, o) in enumerate(zip(solvers, other)):
        o.advance_batch_async(3)
        o.finish_advance_batch()
        assert np.array_equal(s.tree.get_interior().view(np.uint64), o.tree.get_interior().view(np.uint64)), k


def test_autotune_of_a_batch_of_groups(amr):
    """Autotuning a batch of two groups, one of them small, leaves every
    tree's state as it was, and its time covers both."""
    say("case: autotune of a batch of two groups")
    solvers, states = [], []
    rng = np.random.default_rng(9)
    for level in (7, 7, 7, 6):  # 3 x 64 MiB, then 16 MiB that do not fit with them
        t = amr.NdTree(2, 7, 16, 1, 1 << (2 * level))
        solvers.append(amr.AmrSolver(t, (0.5, -1.0), 0.4))
        for _ in range(level):
            t.refine_all()
        states.append(rng.standard_normal(t.size() * t.ni))
        t.set_interior(states[-1])
    alone = amr.Batch([s.tree for s in solvers[:1]])
    batch = amr.Batch([s.tree for s in solvers])
    _, one = alone.autotune(10)
    _, us = batch.autotune(10)
    assert us > 2 * one  # 3.25 times the leaves
    batch.scatter()
    for s, u in zip(solvers, states):
        assert np.array_equal(s.tree.get_interior().reshape(-1), u)
    batch.advance(3)
    batch.scatter()
    for s, u in zip(solvers, states):
        got = s.tree.get_interior()
        s.tree.set_interior(u)
        s.advance_batch_async(3)
        s.finish_advance_batch()
        assert np.array_equal(s.tree.get_interior().view(np.uint64), got.view(np.uint64))
