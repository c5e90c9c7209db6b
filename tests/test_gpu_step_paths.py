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


def test_euler_batch_captured(amr):
    """An Euler batch recorded into a graph on the context's stream and
    replayed, with plain batches in between: finish_advance_batch returns the
    sums of whichever ran last."""
    import torch

    say("case: captured Euler batch")
    made = []
    for _ in range(2):
        s = amr.EulerSolver(2, 6, 16, 1, 72, (1.0, 1.0), 1.4, 0.3)
        for _ in range(2):
            s.tree.refine_all()
        rng = np.random.default_rng(11)
        u0 = np.empty((4, s.tree.size() * s.tree.ni))
        u0[0], u0[1:3], u0[3] = rng.uniform(0.5, 1.5, u0.shape[1]), rng.uniform(-0.5, 0.5, u0[1:3].shape), 3.0
        s.tree.set_interior(u0)
        made.append(s)
    s, plain = made
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(torch.cuda.ExternalStream(s.tree.stream())):
        graph.capture_begin()
        s.advance_batch_async(2)  # recorded, not run
        graph.capture_end()
        for steps in (4, None, None, 6, None, 2, None):
            (s.advance_batch_async(steps) if steps else graph.replay())
            plain.advance_batch_async(steps or 2)
            assert s.finish_advance_batch() == plain.finish_advance_batch(), steps
            assert s.compute_dt() == plain.compute_dt(), steps
            assert_fields(s.tree.get_interior(), plain.tree.get_interior(), f"after {steps}")


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


def euler_step_of_padded(tree, gamma, dt):
    """One Euler step in numpy from the library's padded patches, in the
    expression order of rusanovFlux and time_step_cpu."""
    pad = tree.get_patches()  # [fields, leaves, ...]
    level = (tree.keys() & np.uint64(63)).astype(np.int64)
    cs = tree.cell_sizes(level)
    h, rank = tree.halo, tree.rank
    core = tuple(slice(h, -h) for _ in range(rank))

    def shifted(d, by):
        j = rank - 1 - d
        at = list(core)
        at[j] = slice(h + by, pad.shape[2 + j] - h + by)
        return pad[(slice(None), slice(None), *at)]

    def state(U):
        inv = 1.0 / U[0]
        kin = np.zeros_like(inv)
        for d in range(rank):
            kin = kin + U[1 + d] * U[1 + d]
        kin = kin * (0.5 * inv)
        p = (gamma - 1.0) * (U[rank + 1] - kin)
        return inv, p, np.sqrt(gamma * p * inv)

    def flux(UL, L, UR, Rt, d):
        ul, ur = UL[1 + d] * L[0], UR[1 + d] * Rt[0]
        sl, sr = np.abs(ul) + L[2], np.abs(ur) + Rt[2]
        smax = np.where(sl < sr, sr, sl)
        out = np.empty_like(UL)
        out[0] = 0.5 * (UL[1 + d] + UR[1 + d] - smax * (UR[0] - UL[0]))
        for k in range(rank):
            fl, fr = UL[1 + k] * ul, UR[1 + k] * ur
            if k == d:
                fl, fr = fl + L[1], fr + Rt[1]
            out[1 + k] = 0.5 * (fl + fr - smax * (UR[1 + k] - UL[1 + k]))
        fl, fr = ul * (UL[rank + 1] + L[1]), ur * (UR[rank + 1] + Rt[1])
        out[rank + 1] = 0.5 * (fl + fr - smax * (UR[rank + 1] - UL[rank + 1]))
        return out

    U = pad[(slice(None), slice(None), *core)]
    sU, total = state(U), np.zeros_like(U)
    for d in range(rank):
        lo, hi = shifted(d, -1), shifted(d, 1)
        left, right = flux(lo, state(lo), U, sU, d), flux(U, sU, hi, state(hi), d)
        total -= (dt / cs[:, d]).reshape((1, -1) + (1,) * rank) * (right - left)
    return U + total


# (rank, extents): one strip and several, strips that end early, idle lanes, a
# layer as wide as the workgroup, one too wide for it, and one whose strip is
# too large for LDS (both from memory)
EULER_BOXES = [(2, (2, 2)), (2, (2, 128)), (2, (130, 4)), (2, (32, 32)), (2, (22, 40)), (2, (6, 300)), (2, (4, 516)),
               (3, (2, 2, 2)), (3, (12, 10, 6)), (3, (4, 6, 8)), (3, (6, 16, 16)), (3, (16, 16, 16)), (3, (2, 4, 30)),
               (3, (10, 16, 32)), (3, (4, 24, 24))]


@pytest.mark.parametrize("rank,ext", EULER_BOXES)
def test_any_shape_euler(amr, rank, ext):
    """Euler steps of any-shape patches, one call and a batch, on a tree with
    same-level, finer and coarser faces."""
    say(f"case: any-shape Euler {ext}")
    rng = np.random.default_rng(sum(ext))
    s, batch = (amr.EulerSolver(rank, 4, ext, 1, 200, (1.0,) * rank, 1.4, 0.3) for _ in range(2))
    for t in (s.tree, batch.tree):
        refine_mixed(t)
    t = s.tree
    u0 = np.empty((t.fields, t.size() * t.ni))
    u0[0] = rng.uniform(0.5, 1.5, u0.shape[1])
    u0[1:-1] = rng.uniform(-0.5, 0.5, u0[1:-1].shape)
    u0[-1] = rng.uniform(2.0, 4.0, u0.shape[1])
    for x in (s, batch):
        x.tree.set_interior(u0)
    time = 0.0
    for step in range(3):
        with np.errstate(all="ignore"):  # the corners of the padded patches are 0
            exp = euler_step_of_padded(t, 1.4, s.compute_dt())
        time += s.advance()
        assert_fields(t.get_interior(), exp, f"{ext} step {step}")
    batch.advance_batch_async(3)
    assert batch.finish_advance_batch() == (time, 3)
    assert_fields(batch.tree.get_interior(), t.get_interior(), f"{ext} batch")


@pytest.mark.parametrize("n", [4093, 4096])
def test_euler_walk_16(amr, n):
    """16^2 patches on both sides of the leaf count from which a wave walks a
    leaf."""
    say(f"case: Euler 16^2, {n} leaves")
    s = amr.EulerSolver(2, 7, 16, 1, 4200, (1.0, 1.0), 1.4, 0.3)
    t = s.tree
    for _ in range(6):
        t.refine_all()
    if n < 4096:  # one family coarsened
        flags = np.zeros(t.size(), dtype=np.int8)
        flags[:4] = amr.COARSEN
        assert t.reconstruct_tree(flags)
    assert t.size() == n
    rng = np.random.default_rng(n)
    u0 = np.empty((4, t.size() * t.ni))
    u0[0], u0[1:3], u0[3] = rng.uniform(0.5, 1.5, u0.shape[1]), rng.uniform(-0.5, 0.5, u0[1:3].shape), 3.0
    t.set_interior(u0)
    with np.errstate(all="ignore"):
        exp = euler_step_of_padded(t, 1.4, s.compute_dt())
    s.advance()
    assert_fields(t.get_interior(), exp, f"{t.size()} leaves")


@pytest.mark.parametrize("rank,level", [(2, 5), (2, 6), (3, 3), (3, 4)])
def test_regrid_on_both_sides_of_the_lds_limit(amr, rank, level):
    """Regrids that start and end below, at and above 4096 leaves (keys in LDS
    or in memory), against the oracle: keys and neighbour tables."""
    from oracle import OracleTree

    say(f"case: regrids of a {rank}D tree at level {level}")
    n = 4
    g = amr.NdTree(rank, level + 2, n, 1, 80000)
    o = OracleTree(rank, n, 1, level + 2, 80000)
    for _ in range(level):
        g.refine_all()
        o.refine_all()
    assert g.size() == 1 << (rank * level)
    rng = np.random.default_rng(rank * 10 + level)
    for share in (0.3, 0.05, 0.0):
        flags = np.where(rng.random(g.size()) < share, amr.REFINE, amr.COARSEN).astype(np.int8)
        assert bool(g.reconstruct_tree(flags)) == bool(o.reconstruct(flags))
        assert np.array_equal(g.keys(), o.keys()), share
        assert g.neighbor_metadata().tobytes() == o.metadata().tobytes(), share


def test_adjoint_segments_ride_along(amr):
    """2D 16^2 gradients whose recomputed segments share the adjoint steps'
    launches: the same bits for every checkpoint interval (1: nothing to
    recompute; 7: a short last segment; 23: one segment, nothing to share),
    with regrids inside and between segments, first pass and replay."""
    import torch

    say("case: 2D adjoint, checkpoint intervals")
    want = None
    for keep in (23, 1, 2, 5, 7, 22):
        g = amr.NdTree(2, 6, 16, 1, 4100)
        s = amr.AmrSolver(g, (1.0, 0.5), 0.4)
        for _ in range(3):
            g.refine_all()
        s.initialize(lambda c: np.exp(-((c[..., 0] - 0.4) ** 2 + (c[..., 1] - 0.5) ** 2) / (2 * 0.06**2)))
        x = g.get_interior().reshape(-1).copy()
        crit = amr.make_criterion(amr.CRITERION_GRADIENT, 0.01, 0.002, 3, 6)
        tape = amr.Tape(s, 23, crit, 3, keep)
        info = tape.info()
        u0 = torch.from_numpy(x).cuda()
        uT = torch.empty(info["final_leaves"] * info["cells_per_leaf"], dtype=torch.float64, device="cuda")
        lam = torch.from_numpy(np.random.default_rng(6).standard_normal(uT.numel())).cuda()
        grad = torch.empty_like(u0)
        for _ in range(2):
            tape.forward(u0.data_ptr(), (0.9, -0.4), uT.data_ptr())
            gv = tape.adjoint(lam.data_ptr(), grad.data_ptr())
            got = (uT.cpu().numpy(), grad.cpu().numpy(), gv)
            if want is None:
                want = got
                assert info["topologies"] > 2, info
            for a, b in zip(got, want):
                assert np.array_equal(a, b), keep


# (rank, extents): smallest, uneven, tiles that just fit in LDS and just do not
ADJOINT_BOXES = [(2, (2, 2)), (2, (12, 8)), (2, (62, 62)), (2, (62, 64)), (2, (6, 300)), (3, (2, 2, 2)),
                 (3, (12, 10, 6)), (3, (14, 14, 14)), (3, (14, 14, 16))]


@pytest.mark.parametrize("rank,ext", ADJOINT_BOXES)
def test_any_shape_adjoint(amr, rank, ext):
    """One step of any-shape patches is linear in u and, with dt and the signs
    of v fixed, in v: the adjoint satisfies the dot-product identity and
    grad_v is the central difference of any width, both up to rounding (a few
    ulp of each of the products summed, over the width)."""
    import math

    import torch

    say(f"case: any-shape adjoint {ext}")
    vel = (0.8, -0.5, 0.25)[:rank]
    g = amr.NdTree(rank, 4, ext, 1, 200)
    s = amr.AmrSolver(g, vel, 0.4)
    refine_mixed(g)
    rng = np.random.default_rng(sum(ext))
    u0, lam = rng.standard_normal((2, g.size() * g.ni))
    g.set_interior(u0)
    tape = amr.Tape(s, 1, None, 0, 1)
    u, l = torch.from_numpy(u0).cuda(), torch.from_numpy(lam).cuda()
    out, grad = torch.empty_like(u), torch.empty_like(u)

    def image(v):
        tape.forward(u.data_ptr(), v, out.data_ptr())
        return math.fsum(lam * out.cpu().numpy())

    lhs = image(vel)
    gv = tape.adjoint(l.data_ptr(), grad.data_ptr())
    scale = np.linalg.norm(u0) * np.linalg.norm(lam)
    assert abs(lhs - math.fsum(u0 * grad.cpu().numpy())) <= 1e-13 * scale
    h = 0.125
    for d in range(rank):
        lo, hi = list(vel), list(vel)
        lo[d] -= h
        hi[d] += h
        fd = (image(hi) - image(lo)) / (2 * h)
        assert abs(fd - gv[d]) <= 1e-13 * scale / h, (d, fd, gv[d])


def test_tape_memory_follows_the_checkpoint_interval(amr):
    """A tape of a large 2D 16^2 tree holds one segment of states besides its
    checkpoints and work buffers, and its gradient is the same bits as with
    every state kept."""
    import torch

    say("case: tape of 16384 leaves")
    n, steps, keep = 16384, 24, 12
    g = amr.NdTree(2, 7, 16, 1, n)
    s = amr.AmrSolver(g, (1.0, 0.5), 0.4)
    for _ in range(7):
        g.refine_all()
    assert g.size() == n
    x = np.random.default_rng(2).standard_normal(n * g.ni)
    u0, lam = torch.from_numpy(x).cuda(), torch.from_numpy(x[::-1].copy()).cuda()
    uT, grad = torch.empty_like(u0), torch.empty_like(u0)
    results = []
    for every in (keep, steps):
        g.set_interior(x)
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        tape = amr.Tape(s, steps, None, 0, every)
        used = before - torch.cuda.mem_get_info()[0]
        state = n * g.ni * 8
        # the segment's states, the checkpoints, lambda twice and one more state
        assert used < (every - 1 + -(-steps // every) + 3 + 2) * state, (every, used / state)
        tape.forward(u0.data_ptr(), (0.9, -0.4), uT.data_ptr())
        gv = tape.adjoint(lam.data_ptr(), grad.data_ptr())
        results.append((uT.cpu().numpy(), grad.cpu().numpy(), gv))
        tape.close()
    for a, b in zip(*results):
        assert np.array_equal(a, b)


def test_euler_walk_16_adapted(amr):
    """16^2 patches above the leaf count from which a wave walks a leaf, with
    finer and coarser faces: a step against numpy, then a batch (which folds
    each next dt) against single steps."""
    say("case: Euler 16^2, 4102 leaves on two levels")
    made = []
    for _ in range(2):
        s = amr.EulerSolver(2, 7, 16, 1, 4200, (1.0, 1.0), 1.4, 0.3)
        t = s.tree
        for _ in range(6):
            t.refine_all()
        flags = np.zeros(t.size(), dtype=np.int8)
        flags[[0, 2741]] = amr.REFINE
        assert t.reconstruct_tree(flags) and t.size() == 4102
        rng = np.random.default_rng(16)
        u0 = np.empty((4, t.size() * t.ni))
        u0[0], u0[1:3], u0[3] = rng.uniform(0.5, 1.5, u0.shape[1]), rng.uniform(-0.5, 0.5, u0[1:3].shape), 3.0
        t.set_interior(u0)
        made.append(s)
    single, batch = made
    with np.errstate(all="ignore"):  # the corners of the padded patches are 0
        exp = euler_step_of_padded(single.tree, 1.4, single.compute_dt())
    time = single.advance()
    assert_fields(single.tree.get_interior(), exp, "one step")
    for _ in range(2):
        time += single.advance()
    batch.advance_batch_async(3)
    assert batch.finish_advance_batch() == (time, 3)
    assert_fields(batch.tree.get_interior(), single.tree.get_interior(), "batch of three")
