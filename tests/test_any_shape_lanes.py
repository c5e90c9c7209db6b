"""The any-shape kernels themselves -- walks, index arithmetic, LDS, barriers --
run on the CPU lane by lane (tests/cpp/any_shape_lanes.cpp), under the
compiler's address and undefined-behaviour checks and with every array of its
exact size: against the item bodies that the emulation tests pin to the oracle,
and for the Euler equations a step in numpy, bit for bit (neither side
contracts; the adjoint's velocity sums, whose order differs, to the rounding of
a sum)."""
import os
import subprocess
import types

import numpy as np
import pytest

import emulation as emu
from oracle import OracleTree
from test_gpu_step_paths import euler_step_of_padded

DEPTH = 4
BIN = emu.HERE / "cpp" / "any_shape_lanes.bin"


@pytest.fixture(scope="module", autouse=True)
def built():
    subprocess.run(["make", "-s", "-C", str(emu.HERE / "cpp"), str(BIN)], check=True, capture_output=True)


def mixed(rank):
    """Keys and tables of a tree with faces of all three relations on every
    side: level 1 with its first leaf refined, and in that family the last
    again."""
    o = OracleTree(rank, 4, 1, DEPTH, 400)
    o.refine_all()
    for leaf in (0, (1 << rank) - 1):
        flags = np.zeros(o.size(), dtype=np.int8)
        flags[leaf] = 1
        assert o.reconstruct(flags)
    keys = o.keys()
    links, metas, err = emu.build_table(rank, DEPTH, keys)
    assert err == 0
    return keys, links, metas


def lanes(tmp_path, kind, rank, ext, table, arrays, reverse=0, count=None):
    keys, links, metas = table
    head = np.array([kind, rank, *(list(ext) + [1] * (3 - rank)), keys.size, reverse, count or keys.size], np.int32)
    with open(tmp_path / "in", "wb") as f:
        for a in (head, keys, links, metas, *(np.asarray(x, dtype=np.float64) for x in arrays)):
            f.write(np.ascontiguousarray(a).tobytes())
    r = subprocess.run([str(BIN), str(tmp_path / "in"), str(tmp_path / "out")], capture_output=True, text=True,
                       env={**os.environ, "ASAN_OPTIONS": "verify_asan_link_order=0:detect_leaks=0"})
    assert r.returncode == 0, r.stderr[-3000:]
    return np.fromfile(tmp_path / "out", dtype=np.float64)


def same(a, b):
    a, b = np.ascontiguousarray(a).reshape(-1), np.ascontiguousarray(b).reshape(-1)
    assert a.size == b.size
    bad = np.flatnonzero(a.view(np.uint64) != b.view(np.uint64))
    assert bad.size == 0, (bad.size, bad[:5], a[bad[:5]], b[bad[:5]])


# one pass and several, partial last pass, a layer as wide as the workgroup and
# wider, more ghost items than threads, the smallest patch, tiles that just fit
# in LDS and that just do not
STEP = [(2, 2), (2, 128), (130, 4), (6, 300), (90, 88), (94, 94), (62, 64), (2, 2, 2), (12, 10, 6), (6, 16, 16),
        (4, 18, 20), (2, 4, 30), (4, 24, 24)]


@pytest.mark.parametrize("ext", STEP, ids=str)
def test_advection_step(tmp_path, ext):
    rank = len(ext)
    table = keys, links, metas = mixed(rank)
    n = keys.size * int(np.prod(ext))
    vel = (1.0, -0.5, 0.25)[:rank]
    u = np.random.default_rng(sum(ext)).standard_normal(n)
    dtdx, v, hs = emu.step_params(rank, ext, DEPTH, 3, vel, 1e-3)
    got = lanes(tmp_path, 0, rank, ext, table, (v, hs, dtdx, u), reverse=sum(ext) // 2 % 2)
    same(got, emu.step_box(rank, ext, keys, links, metas, u, dtdx, v, hs))


@pytest.mark.parametrize("ext", [(2, 2), (12, 8), (62, 62), (62, 64), (6, 300), (2, 2, 2), (12, 10, 6), (14, 14, 14),
                                 (14, 14, 16)], ids=str)
def test_adjoint_step(tmp_path, ext):
    rank = len(ext)
    table = keys, links, metas = mixed(rank)
    n = keys.size * int(np.prod(ext))
    vel = np.array((0.8, -0.5, 0.25)[:rank] + (0.0,) * (3 - rank))
    lam, u = np.random.default_rng(sum(ext)).uniform(-1.0, 1.0, (2, n))
    dtdx, _, _ = emu.step_params(rank, ext, DEPTH, 3, vel[:rank], 1e-3)
    vp, vm = 0.5 * (vel + np.abs(vel)), 0.5 * (vel - np.abs(vel))
    got = lanes(tmp_path, 1, rank, ext, table, (dtdx, vp, vm, np.sign(vel), lam, u))
    want, sums = emu.adj_step_box(rank, ext, keys, links, metas, lam, u, dtdx, vel[:rank])
    same(got[: lam.size], want)
    # |term| <= 2 dt/dx with |lambda|, |u| <= 1; n of them, each partial sum rounded
    bound = 2.0 * dtdx.max() * np.prod(ext) ** 2 * np.finfo(float).eps
    assert np.abs(got[lam.size :].reshape(sums.shape) - sums).max() <= bound


# one strip and several, strips that end early, idle lanes, a layer as wide as
# the workgroup, one too wide for it, and one whose strip is too large for LDS;
# split for the tree's own leaves (short strips) or for many (long ones)
EULER = [((2, 2), 0), ((2, 16), 0), ((2, 128), 0), ((2, 128), 100000), ((130, 4), 0), ((32, 32), 0), ((32, 32), 100000),
         ((22, 40), 0), ((22, 40), 100000), ((6, 300), 0), ((4, 48), 0), ((4, 48), 100000), ((4, 516), 0),
         ((16, 16), 100000), ((2, 2, 2), 0), ((12, 10, 6), 0), ((12, 10, 6), 100000), ((4, 6, 8), 0),
         ((4, 6, 8), 100000), ((6, 16, 16), 0), ((2, 4, 30), 0), ((2, 4, 30), 100000), ((4, 24, 24), 0),
         ((6, 6, 6), 0), ((6, 6, 6), 100000)]


@pytest.mark.parametrize("ext,count", EULER, ids=str)
def test_euler_step(tmp_path, ext, count):
    rank = len(ext)
    gamma, cfl = 1.4, 0.3
    table = keys, links, metas = mixed(rank)
    n = keys.size * int(np.prod(ext))
    rng = np.random.default_rng(sum(ext))
    u = np.empty((rank + 2, n))
    u[0], u[1:-1], u[-1] = rng.uniform(0.5, 1.5, n), rng.uniform(-0.5, 0.5, (rank, n)), rng.uniform(2.0, 4.0, n)
    cs = np.zeros((17, 3))
    for lv in range(DEPTH + 1):
        for d in range(rank):
            cs[lv, d] = (float(1 << (DEPTH - lv)) / float(1 << DEPTH)) / float(ext[rank - 1 - d])
    level = (keys & np.uint64(63)).astype(int)

    def dt_of(u):
        U = u.reshape(rank + 2, keys.size, -1)
        inv = 1.0 / U[0]
        kin = np.zeros_like(inv)
        for d in range(rank):
            kin = kin + U[1 + d] * U[1 + d]
        p = (gamma - 1.0) * (U[-1] - kin * (0.5 * inv))
        a = np.sqrt(gamma * p * inv)
        return cfl * min((cs[level, d][:, None] / (np.abs(U[1 + d] * inv) + a)).min() for d in range(rank))

    tree = types.SimpleNamespace(
        halo=1, rank=rank, keys=lambda: keys, cell_sizes=lambda lv: cs[lv, :rank],
        get_patches=lambda: np.stack([emu.padded_box(rank, ext, 1, links, metas, f, keys.size) for f in u]))
    got = lanes(tmp_path, 2, rank, ext, table, ((gamma, cfl), cs, u), reverse=sum(ext) // 2 % 2, count=count)
    with np.errstate(all="ignore"):  # the corners of the padded patches are 0
        want = euler_step_of_padded(tree, gamma, dt_of(u))
    same(got[: u.size], want)
    same(got[u.size : u.size + 2], np.array([dt_of(u), dt_of(want)]))


def test_walks_cover_every_patch():
    """The split of a patch that the host chooses, over the shapes that the
    library takes and few to many leaves: it ends, its lanes, passes, strips
    and groups cover every layer once, and it keeps to the LDS limit."""
    shapes = [(a, b) for a in (*range(2, 70, 2), 126, 128, 130, 500, 1000, 4096) for b in (*range(2, 70, 2), 128, 190,
              192, 194, 256, 258, 510, 512, 514, 4096)]
    shapes += [(a, b, c) for a in (2, 4, 6, 8, 10, 14, 30, 64, 256) for b in (2, 4, 6, 8, 12, 16, 22, 32)
               for c in (2, 4, 6, 8, 10, 16, 20, 24, 30, 32, 64)]
    for ext in shapes:
        cols = int(np.prod(ext[1:]))
        for leaves in (1, 7, 100, 1023, 5000, 100000):
            (sl, passes, st), (segs, layers, groups, et, lds) = emu.walks(len(ext), ext, leaves)
            if st:
                assert sl * cols <= st and sl * (passes - 1) < ext[0] <= sl * passes, ext
            else:
                assert cols > 256, ext
            if et:
                assert segs * cols <= et and lds <= 65536 and min(segs, layers, groups) >= 1, ext
                assert segs * layers * (groups - 1) < ext[0] <= segs * layers * groups, (ext, leaves)
            else:
                # LDS, or leaves times strips beyond the division by multiplication
                assert cols > 128 or leaves * (ext[0] // 4 + 1) ** 2 >= 1 << 32, (ext, leaves)
