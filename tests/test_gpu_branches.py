"""GPU kernels at the sizes where their dispatch changes, against the oracle.

Each test drives one kernel family over the edges of its size classes (lanes
per item, rows per workgroup, rounds of a loop); bars are those of the parity
tests of the same stage.
"""
import numpy as np
import pytest

from sw_reaxff_amd import systems

from .parity import harness
from .test_bonded import _gpu_vs_oracle as _gpu_bonded_vs_oracle
from .test_valence import _gpu_tor_vs_oracle, _gpu_vs_oracle


def lattice(m=8, a=1.7, seed=3):
    """m^3 C/H/O atoms on a shaken cubic lattice: every atom has a dozen or
    more bonds, so centres have up to 135 angles and bonds up to 99
    quadruples (more than one round of a 64-lane group)."""
    rng = np.random.default_rng(seed)
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3) * a
    x = g + rng.normal(scale=0.05, size=g.shape) + 20.0
    t = rng.integers(1, 4, size=len(x)).astype(np.int32)
    return systems.System(x=x, v=np.zeros_like(x), type=t, tag=np.arange(1, len(x) + 1, dtype=np.int32),
                          elements=["H", "O", "C"], lo=np.zeros(3), hi=np.full(3, 60.0), periodic=False)


GROUP_SYSTEMS = {
    "lattice": lambda: lattice(),                         # items of 1 to more than 64 evaluations
    "cluster21": lambda: systems.cluster(20, seed=1),     # 21 centres, 28 bonds: one or two waves
    "water4200": lambda: systems.water_box(1400, seed=4),   # 4,200 centres: past the 16-lane minimum
    "water30k": lambda: systems.water_box(10000, seed=5),   # 30,000 centres, ~17,600 bonds: single lanes
}


@pytest.mark.gpu
@pytest.mark.parametrize("case", list(GROUP_SYSTEMS))
def test_gpu_valence_and_torsion_groups(gpu_lib, oracle_lib, ffield, case):
    s = GROUP_SYSTEMS[case]()
    for check in (_gpu_vs_oracle, _gpu_tor_vs_oracle):
        check(oracle_lib, ffield, harness(s, ffield, tol=1e-10), s.elements, s.type, s.tag)


def shuffled(s, seed):
    """s with its atoms in random order: a workgroup's atoms share no partners."""
    k = np.random.default_rng(seed).permutation(s.n)
    return systems.System(x=s.x[k], v=s.v[k], type=s.type[k], tag=np.arange(1, s.n + 1, dtype=np.int32),
                          elements=s.elements, lo=s.lo, hi=s.hi, periodic=s.periodic)


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["lattice", "cluster21", "water4200", "water30k", "shuffled36k"])
def test_gpu_bonded_groups(gpu_lib, oracle_lib, ffield, case):
    """Atom energies, hydrogen bonds and dBond forces: atoms with more bonds
    than their four lanes and more than 64 hydrogen-bond entries (lattice),
    workgroups of 8, 16 and 64 atoms in the hydrogen-bond pass, and one whose
    partners overfill its LDS table (shuffled)."""
    s = shuffled(systems.water_box(12000, seed=7), 8) if case == "shuffled36k" else GROUP_SYSTEMS[case]()
    _gpu_bonded_vs_oracle(gpu_lib, oracle_lib, ffield, harness(s, ffield, tol=1e-10), s.elements, s.type, s.tag)


def waters(m, seed):
    """A non-periodic cluster of m waters (3 m atoms)."""
    s = systems.water_box(m, seed=seed)
    return systems.System(x=s.x, v=s.v, type=s.type, tag=s.tag, elements=s.elements, lo=s.x.min(0) - 12.0,
                          hi=s.x.max(0) + 12.0, periodic=False)


@pytest.mark.gpu
def test_gpu_small_cg_takes_the_general_solves_bits(gpu_lib, ffield):
    """1024 panels in all is the most the one-launch-per-iteration solve takes;
    with one more one-panel system the general solve runs instead.  Systems of
    1 to 3072 rows around the panel (64) and tile (256) edges: the charges
    and iteration counts of the common systems are the same bits."""
    from sw_reaxff_amd.batch import Batch
    parts = [waters(m, seed=m) for m in (1024, 86, 85, 22, 21)] + [waters(1, seed=100 + k) for k in range(964)]
    assert sum(-(-s.n // 64) for s in parts) == 1024
    got = []
    for extra in ([], [waters(1, seed=2000)]):
        bt = Batch(ffield, tol=1e-6)
        bt.load(parts + extra)
        bt.evaluate()
        bt.sync()
        n = int(bt.packed.row_off[len(parts)])
        got.append((bt.sys.get("q")[:n], bt.iterations()[:len(parts)]))
    assert got[0][1].max() > 10
    assert np.array_equal(got[0][0], got[1][0])
    assert np.array_equal(got[0][1], got[1][1])


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 21, 22, 85, 86, 1024, 1025])
def test_gpu_cg_sizes_against_oracle(gpu_lib, oracle_lib, ffield, m):
    """One system of 3 m rows, up to the last small and the first general one."""
    from .parity import atoms_of, make_oracle
    s = waters(m, seed=m)
    lmp = harness(s, ffield, tol=1e-10)
    h = lmp.system
    h.sync()
    o = make_oracle(oracle_lib, ffield, s.elements, atoms_of(h), tol=1e-10)
    o.build_verlet(12.0)
    o.step()
    assert np.max(np.abs(h.get("q")[:s.n] - o.get("q")[:s.n])) <= 1e-9


@pytest.mark.gpu
def test_gpu_tiny_cg_takes_the_small_solves_bits(gpu_lib, ffield):
    """Systems of 3 to 64 rows, solved in one launch; with the last two declared
    one system of 120 rows the batch takes a launch per iteration: the others'
    charges and iteration counts are the same bits, in a first solve and from its
    history."""
    import ctypes as C

    from sw_reaxff_amd import _lib
    from sw_reaxff_amd.batch import Batch
    w = waters(22, seed=8)
    cut = systems.System(x=w.x[:64], v=w.v[:64], type=w.type[:64], tag=w.tag[:64], elements=w.elements, lo=w.lo,
                         hi=w.hi, periodic=False)
    parts = [waters(1, seed=1), waters(7, seed=2), systems.cluster(20, seed=1), waters(21, seed=3), cut,
             waters(20, seed=4), waters(20, seed=5)]
    assert [s.n for s in parts] == [3, 21, 21, 63, 64, 60, 60]
    got = []
    for merge in (False, True):
        bt = Batch(ffield, tol=1e-6)
        P = bt.load(parts)
        off = np.ascontiguousarray(np.delete(P.row_off, -2) if merge else P.row_off, dtype=np.int32)
        h = bt.sys
        _lib.check(h.L.swr_set_batch(h.h, off.size - 1, off.ctypes.data_as(C.POINTER(C.c_int))), "swr_set_batch")
        h.build_neighbors(10.0)
        n = int(P.row_off[5])
        for _ in range(3):
            h.call("qeq_init_matvec")
            h.qeq_cg()
            h.call("calculate_q")
            h.sync()
            got.append((merge, h.get("q")[:n], h.get("sys_iters").reshape(-1, 2)[:5].copy()))
    for a, b in zip(got[:3], got[3:]):
        assert np.array_equal(a[1], b[1]) and np.array_equal(a[2], b[2])
    assert got[0][2].max() > 10


@pytest.mark.gpu
@pytest.mark.parametrize("m", [20, 30])
def test_gpu_small_cg_with_an_empty_system(gpu_lib, ffield, m):
    """A batch may hold systems without rows: nothing waits for them (60 rows:
    one launch for the solve; 90: one per iteration)."""
    import ctypes as C

    from sw_reaxff_amd import _lib
    s = waters(m, seed=3)
    got = []
    for off in ([0, s.n], [0, 0, s.n, s.n]):
        h = _lib.System(ffield, s.elements, tol=1e-6)
        h.set_atoms(s.n, s.x, s.type, s.tag)
        o = np.array(off, dtype=np.int32)
        _lib.check(h.L.swr_set_batch(h.h, len(off) - 1, o.ctypes.data_as(C.POINTER(C.c_int))), "swr_set_batch")
        h.build_neighbors()
        h.call("qeq_init_matvec")
        its = h.qeq_cg()
        h.call("calculate_q")
        h.sync()
        got.append((its, h.get("q")[:s.n]))
    assert got[0][0] == got[1][0] and got[0][0][0] < 100
    assert np.array_equal(got[0][1], got[1][1])


@pytest.mark.gpu
@pytest.mark.parametrize("m,a", [(8, 1.7), (10, 1.7), (21, 1.7)])
def test_gpu_bond_marks_of_crowded_ghosts(gpu_lib, ffield, m, a):
    """sort_bonds_C's one in-order pass restated over the GPU's own bond lists,
    where ghosts have a dozen bonds: the search with its neighbour lists in
    LDS (10,000 ghosts), in memory (13,000) and the relaxation (34,000)."""
    from sw_reaxff_amd import _lib
    s = lattice(m, a, seed=m)
    x = np.mod(s.x - 20.0, m * a)
    xa, owner = systems.borders(x, np.zeros(3), np.full(3, m * a), 12.0)
    h = _lib.System(ffield, s.elements)
    h.set_atoms(s.n, xa, s.type[owner], s.tag[owner], owner=owner)
    h.build_neighbors()
    h.set_capacities(np.full(owner.size, 32), np.full(owner.size, 256))
    for stage in ("write_reax_atoms_and_pack", "reset", "write_reax_lists_init_forces", "validate_lists", "sort_bonds"):
        h.call(stage)
    h.sync()
    n, N = s.n, owner.size
    bi, be, nbr = h.get("bond_index"), h.get("bond_end"), h.get("bonds")["nbr"]
    mark = np.full(N, 1000)
    mark[:n] = 0
    most = 0
    for i in range(n, N):
        j = nbr[bi[i]:be[i]]
        most = max(most, int((j > i).sum()), int((j < i).sum()))
        if j.size:
            mark[i] = min(mark[i], (mark[j] + 1).min())
    assert most > 8 and (mark[n:] < 1000).any()
    assert {8: N - n <= 12288, 10: 12288 < N - n <= 32512, 21: N - n > 32512}[m]
    assert np.array_equal(h.get("bond_mark")[:N], mark)


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["water1000", "cluster21", "lattice", "no_hydrogen", "overfull"])
def test_gpu_first_lists_from_the_estimate_pass(gpu_lib, ffield, case):
    """New atoms' lists come from the capacity estimate's far pass: the same
    bits as Reset and the fused pass stage by stage, and the same refusal when
    an atom has more bond candidates than the pass keeps."""
    from sw_reaxff_amd import _lib
    s = {"water1000": lambda: systems.water_box(333, seed=6), "cluster21": lambda: systems.cluster(20, seed=1),
         "lattice": lattice, "no_hydrogen": lattice, "overfull": lambda: lattice(8, 0.9)}[case]()
    if case == "no_hydrogen":
        s.type[:] = np.where(s.type == 1, 2, s.type)
    got = []
    for stages in (("pair_compute",), ("write_reax_atoms_and_pack", "reset", "write_reax_lists_init_forces",
                                       "validate_lists", "sort_bonds", "bo")):
        h = _lib.System(ffield, s.elements)
        xa, owner = systems.borders(s.x, s.lo, s.hi, 12.0) if s.periodic else (s.x, np.arange(s.n))
        h.set_atoms(s.n, xa, s.type[owner], s.tag[owner], owner=owner)
        h.build_neighbors()
        try:
            for stage in stages:
                h.call(stage)
            h.sync()
            out = {k: h.get(k) for k in ("far_index", "far_end", "num_bonds", "num_hbonds", "Hindex", "bond_index",
                                         "bond_end", "bonds", "BO", "bo_data")}
            numH = int((out["Hindex"] >= 0).sum())
            assert (numH == 0) == (case == "no_hydrogen")
            for k in ("hbond_index", "hbond_end"):
                out[k] = h.get(k)[:numH]
            rows = [np.concatenate([np.zeros(0, int)] + [np.arange(a, b) for a, b in zip(out[k + "_index"], out[k + "_end"])])
                    for k in ("bond", "hbond")]
            for k in ("bonds", "BO", "bo_data"):
                out[k] = out[k][rows[0]]
            rows, hb = rows[1], h.get("hbonds")
            out["hb"] = (hb["nbr"][rows], hb["scl"][rows], h.get("hbond_far")[rows])
            assert (rows.size > 0) == (numH > 0)
            got.append(out)
        except _lib.SwrError as e:
            got.append(e.code)
    a, b = got
    assert isinstance(a, int) == isinstance(b, int) == (case == "overfull")
    if case == "overfull":
        assert a == b
        return
    for k in a:
        for x, y in zip(a[k] if k == "hb" else [a[k]], b[k] if k == "hb" else [b[k]]):
            assert x.tobytes() == y.tobytes(), k


@pytest.mark.gpu
@pytest.mark.parametrize("mixed", [0, 1])
@pytest.mark.parametrize("m", [216, 1400])
def test_gpu_charges_queued_behind_the_solve(gpu_lib, ffield, m, mixed):
    """swr_qeq_pre_force queues the charges before it knows that the solve has
    finished: the same bits as solve and charges one after the other, cold
    (several batches of iterations), warm, and when the extrapolated start
    already meets the test (648 atoms: the small solve; 4,200: the general)."""
    from sw_reaxff_amd import _lib
    s = systems.water_box(m, seed=m)
    xa, owner = systems.borders(s.x, s.lo, s.hi, 12.0)
    hs = []
    for _ in range(2):
        h = _lib.System(ffield, s.elements, qeq_mixed=mixed)
        h.set_atoms(s.n, xa, s.type[owner], s.tag[owner], owner=owner)
        h.build_neighbors()
        hs.append(h)
    iters = []
    for rep in range(8):
        out = []
        for k, h in enumerate(hs):
            if rep == 7:   # a start that is the last solution
                for name in ("s_hist", "t_hist"):
                    a = h.get(name).reshape(-1, 5)
                    h.put(name, np.repeat(a[:, :1], 5, axis=1))
            if k == 0:
                its = [_lib.C.c_int(), _lib.C.c_int()]
                h.call("qeq_pre_force", *map(_lib.C.byref, its))
                its = tuple(i.value for i in its)
            else:
                h.call("qeq_init_matvec")
                its = tuple(h.qeq_cg())
                h.call("calculate_q")
            out.append((its, h.scalar("mixed_outer"), h.get("q").tobytes(), h.get("s_hist").tobytes(),
                        h.get("t_hist").tobytes()))
        assert out[0] == out[1]
        iters.append(out[0][:2])
    assert max(iters[0][0]) > (3 if mixed else 16) and max(iters[-1][0]) < max(iters[0][0])
    if mixed:
        assert iters[0][1] > 1 and iters[-1][1] == 1


@pytest.mark.gpu
@pytest.mark.parametrize("n", [2, 1023, 1024, 1025, 16384, 16385])
def test_gpu_reset_and_scans_at_tile_edges(gpu_lib, ffield, n):
    """Reset's positions and the Verlet offsets are the exclusive sums of their
    counts, around one tile of 1,024 atoms and around the 16 tiles that a scan
    takes in one launch; ragged capacities."""
    from sw_reaxff_amd import _lib
    s = systems.water_box(5462, seed=2)
    x, t, tag = s.x[:n], s.type[:n], s.tag[:n]
    rng = np.random.default_rng(n)
    nb, nh = (rng.integers(25, 70, size=n).astype(np.int32) for _ in range(2))
    h = _lib.System(ffield, s.elements)
    h.set_atoms(n, x, t, tag, owner=np.arange(n))
    h.build_neighbors(9.0)
    off = h.get("verlet_offsets")
    assert off.size == n + 1 and off[0] == 0 and h.get("verlet_list").size == off[-1]
    rows, counts = [], []
    for i in {0, n // 2, n - 1}:
        d = ((x - x[i]) ** 2).sum(1)
        rows.append(i)
        counts.append(int((d <= 9.0 ** 2).sum()) - 1)
    assert [int(off[i + 1] - off[i]) for i in rows] == counts
    h.set_capacities(nb, nh)
    for _ in range(2):   # the second one finds the lists sized
        h.call("write_reax_atoms_and_pack")
        h.call("reset")
    h.sync()
    is_h = t == 1 + s.elements.index("H")
    excl = lambda c: np.concatenate([[0], np.cumsum(c)])
    assert h.scalar("numH") == is_h.sum() and h.scalar("total_bonds") == nb.sum()
    assert np.array_equal(h.get("bond_index")[:n], excl(nb)[:-1])
    assert np.array_equal(h.get("bond_end")[:n], excl(nb)[:-1])
    assert np.array_equal(h.get("Hindex")[:n], np.where(is_h, excl(is_h)[:-1], -1))
    assert np.array_equal(h.get("hbond_index"), excl(nh[is_h])[:-1])
    assert np.array_equal(h.get("hbond_end"), excl(nh[is_h])[:-1])
    assert not h.get("fCdDelta")[:n].any()


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 7, 16384, 16385])
def test_gpu_set_atoms_uploads(gpu_lib, ffield, n):
    """The one-upload path (16,384 atoms at most) and the one beyond it put the
    same arrays, with and without charges, owners and images, after a larger
    and after a smaller set."""
    from sw_reaxff_amd import _lib
    rng = np.random.default_rng(n)
    h = _lib.System(ffield, ["H", "O", "C"])
    for m in (n, max(1, n // 3), n):
        nloc = (m + 1) // 2
        x = rng.normal(size=(m, 3)) * 20.0
        t = rng.integers(1, 4, size=m).astype(np.int32)
        tag = rng.permutation(m).astype(np.int32) + 1
        for q, owner, img in ((None, True, None), (rng.normal(size=m), True, True), (None, False, True)):
            k = nloc if owner else m
            own = np.concatenate([np.arange(k), rng.integers(0, k, size=m - k)]).astype(np.int32)
            im = rng.integers(-1, 2, size=(m, 3)).astype(np.int8) if img else None
            h.set_atoms(k, x, t, tag, owner=own if owner else None, img=im, q=q)
            assert np.array_equal(h.get("x")[:3 * m].reshape(-1, 3), x)
            for name, want in (("type", t), ("tag", tag), ("owner", own), ("q", np.zeros(m) if q is None else q),
                               ("img", np.zeros(3 * m, np.int8) if im is None else im.ravel())):
                assert np.array_equal(h.get(name)[:want.size], want), name
    bad = np.full(n, n, np.int32)
    if n > 1:
        with pytest.raises(_lib.SwrError, match="owner out of range"):
            h.set_atoms(n // 2, x, t, tag, owner=bad)


@pytest.mark.gpu
def test_gpu_valence_with_many_parameter_sets(gpu_lib, oracle_lib, ffield, tmp_path):
    """Three parameter sets for H-O-H and H-C-H and five for H-C-O, more than the usual two that the
    valence pass's smaller form has room for."""
    lines = open(ffield).read().splitlines()
    k = next(i for i, l in enumerate(lines) if "Nr of angles" in l)
    n = int(lines[k].split()[0])
    extra = []
    for l in lines[k + 1:k + 1 + n]:
        t = l.split()
        sets = {"232": 3, "212": 3, "213": 5, "312": 5}.get("".join(t[:3]), 1)   # (at most 3 where both ends are alike)
        for m in range(1, sets):
            extra.append("  ".join(t[:3] + [f"{float(t[3]) + 4.0 * m:.4f}", f"{float(t[4]) * (1.0 - 0.15 * m):.4f}"] + t[5:]))
    assert len(extra) == 8
    lines[k] = lines[k].replace(str(n), str(n + len(extra)), 1)
    path = str(tmp_path / "ffield.sets")
    with open(path, "w") as f:
        f.write("\n".join(lines[:k + 1 + n] + extra + lines[k + 1 + n:]) + "\n")
    s = systems.cluster(700, seed=9)
    h = harness(s, path, tol=1e-10)
    _gpu_vs_oracle(oracle_lib, path, h, s.elements, s.type, s.tag)
    plain = harness(s, ffield, tol=1e-10)
    plain.system.call("valence_angles")
    plain.system.sync()
    assert plain.system.get("valence_energy")[0] != h.system.get("valence_energy")[0]


@pytest.mark.gpu
def test_gpu_torsions_of_a_large_batch(gpu_lib, ffield):
    """131,072 atoms and more take the torsion pass's form with two waves a SIMD:
    each member's energies are those of a batch of three (whose other members
    put it elsewhere in the box: coordinates of ~1e3 A round at 1e-13)."""
    from sw_reaxff_amd.batch import Batch
    kinds = [systems.cluster(m, seed=m) for m in (60, 75, 90)]
    got = []
    for reps in (1, 131072 // sum(k.n for k in kinds) + 1):
        bt = Batch(tol=1e-6)
        parts = kinds * reps
        bt.load(parts)
        bt.evaluate(nonbonded=False, bonded=True)
        n = bt.sys.scalar("n")
        assert (n >= 131072) == (reps > 1)
        got.append([bt.sys.get(k).reshape(-1, n) for k in ("torsion_eatom", "valence_eatom")])
    per = sum(k.n for k in kinds)
    for a, b in zip(*got):
        assert np.abs(a).max() > 1e-3
        for r in (0, 1, b.shape[1] // per - 1):
            assert np.max(np.abs(b[:, r * per:(r + 1) * per] - a)) <= 1e-8 * np.abs(a).max()


@pytest.mark.gpu
@pytest.mark.parametrize("m,K", [(1, 1), (2, 1), (1, 1100), (2, 1100), (4, 1100)])
def test_gpu_cold_solves_of_few_rows_launch_few_iterations(gpu_lib, ffield, m, K):
    """r rows take about r iterations, so a first solve of systems of few rows
    queues rows + 2 of them, not the sixteen of larger ones."""
    from sw_reaxff_amd.batch import Batch
    rng = np.random.default_rng(m)
    s = waters(m, seed=m)
    parts = [systems.System(x=s.x + rng.normal(scale=0.05, size=s.x.shape), v=s.v, type=s.type, tag=s.tag,
                            elements=s.elements, lo=s.lo, hi=s.hi, periodic=False) for _ in range(K)]
    bt = Batch(ffield, tol=1e-6)
    bt.load(parts)
    bt.sys.ktimer_enable()
    bt.evaluate()
    bt.sync()
    _, launches = bt.sys.ktimer_read("cg_iter")
    its = int(bt.iterations().max())
    assert 2 <= its <= s.n + 1
    if K > 1:                               # (one launch for the whole solve otherwise)
        assert its <= launches <= min(16, s.n + 2)


@pytest.mark.gpu
@pytest.mark.parametrize("bins", [(64, 64, 1023), (64, 64, 1024), (220, 220, 220), (1100, 1100, 90)])
def test_gpu_scans_of_large_sparse_grids(gpu_lib, ffield, bins):
    """Two clusters in the far corners of a grid: the bins' prefix sums at the
    edge of the scan's flat form (4,096 tiles of 1,024) and beyond it, where the
    tiles' sums are scanned themselves.  Each cluster's rows are those it has
    alone."""
    from sw_reaxff_amd import _lib
    s = waters(64, seed=3)
    span = np.ptp(s.x, axis=0)
    far = 5.0 * np.array(bins) + 2.5 - span          # bins of 5 A and a bit: exactly this many of them
    x = np.vstack([s.x, s.x + far])
    ty, tag = np.concatenate([s.type, s.type]), np.arange(1, 2 * s.n + 1, dtype=np.int32)

    def rows(n, x, ty, tag):
        h = _lib.System(ffield, s.elements)
        h.set_atoms(n, x, ty, tag)
        h.build_neighbors(10.0)
        h.sync()
        off, lst = h.get("verlet_offsets"), h.get("verlet_list")
        assert off[0] == 0 and off[n] == h.scalar("verlet_total")
        return [np.sort(lst[off[i]:off[i + 1]]) for i in range(n)]

    alone, both = rows(s.n, s.x, s.type, s.tag), rows(2 * s.n, x, ty, tag)
    assert sum(map(len, alone)) > 1000
    for i in range(s.n):
        assert np.array_equal(both[i], alone[i]) and np.array_equal(both[s.n + i], alone[i] + s.n), i


@pytest.mark.gpu
@pytest.mark.parametrize("m", [4, 17, 18])
def test_gpu_bond_marks_around_the_searchs_limit(gpu_lib, ffield, m):
    """Crowded ghosts whose neighbour lists four lanes walk together: the last
    lattice the search takes (27,700 ghosts), the first the relaxation does
    (30,000) and a box smaller than the ghost shell, whose ghosts have many
    images."""
    from sw_reaxff_amd import _lib
    a = 1.7
    s = lattice(m, a, seed=m)
    x = np.mod(s.x - 20.0, m * a)
    xa, owner = systems.borders(x, np.zeros(3), np.full(3, m * a), min(12.0, m * a))
    h = _lib.System(ffield, s.elements)
    h.set_atoms(s.n, xa, s.type[owner], s.tag[owner], owner=owner)
    h.build_neighbors()
    h.set_capacities(np.full(owner.size, 32), np.full(owner.size, 256))
    for stage in ("write_reax_atoms_and_pack", "reset", "write_reax_lists_init_forces", "validate_lists", "sort_bonds"):
        h.call(stage)
    h.sync()
    n, N = s.n, owner.size
    assert {4: N - n < 12288, 17: 24576 < N - n <= 28672, 18: 28672 < N - n <= 32512}[m]
    bi, be, nbr = h.get("bond_index"), h.get("bond_end"), h.get("bonds")["nbr"]
    mark = np.where(np.arange(N) < n, 0, 1000)
    for i in range(n, N):
        j = nbr[bi[i]:be[i]]
        if j.size:
            mark[i] = min(mark[i], (mark[j] + 1).min())
    assert (mark[n:] < 1000).any()
    assert np.array_equal(h.get("bond_mark")[:N], mark)
    h.call("sort_bonds")                     # once more over its own result
    h.sync()
    assert np.array_equal(h.get("bond_mark")[:N], mark)


@pytest.mark.gpu
@pytest.mark.parametrize("m", [2389, 2390, 4000, 8192, 8193])
def test_gpu_bonded_groups_around_their_lines(gpu_lib, oracle_lib, ffield, m):
    """Water boxes on both sides of the lines between workgroups of 8, 16 and 64
    atoms in the hydrogen-bond pass (7,168 and 24,576 atoms), in the range of four
    lanes an angle or torsion at least."""
    s = systems.water_box(m, seed=m)
    h = harness(s, ffield, tol=1e-10)
    _gpu_bonded_vs_oracle(gpu_lib, oracle_lib, ffield, h, s.elements, s.type, s.tag)
    for check in (_gpu_vs_oracle, _gpu_tor_vs_oracle):
        check(oracle_lib, ffield, harness(s, ffield, tol=1e-10), s.elements, s.type, s.tag)


@pytest.mark.gpu
def test_gpu_torsions_at_two_waves(gpu_lib, oracle_lib, ffield):
    """The first box whose torsions are listed to two waves a SIMD (32,769 atoms)."""
    s = systems.water_box(10923, seed=9)
    for check in (_gpu_vs_oracle, _gpu_tor_vs_oracle):
        check(oracle_lib, ffield, harness(s, ffield, tol=1e-10), s.elements, s.type, s.tag)


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [[1400], [1100, 30, 1200], [1100, 1200]])
def test_gpu_solves_done_at_setup_queue_few_iterations(gpu_lib, ffield, sizes):
    """Unmoved atoms with their solution as history: the general solve is done at
    its setup, and the host sees it after a few queued iterations instead of the
    sixteen of a first solve; with one system from zero history the batch goes on."""
    from sw_reaxff_amd.batch import Batch
    parts = [waters(m, seed=m) for m in sizes]
    exact, bt = Batch(ffield, tol=1e-9), Batch(ffield, tol=1e-6)
    exact.load(parts)
    exact.evaluate()
    exact.sync()
    hist = [exact.save_history(k, fill=True) for k in range(len(parts))]
    exact.sync()
    bt.sys.ktimer_enable()

    def solve(h):
        bt.load(parts, hist=h)
        bt.sys.ktimer_read("cg_iter", True)
        bt.evaluate()
        bt.sync()
        return bt.sys.ktimer_read("cg_iter")[1], bt.iterations().copy(), [q.copy() for q in bt.charges()]

    launches, its, q = solve(hist)
    assert its.max() == 1 and launches <= 6
    assert all(np.max(np.abs(a - b)) <= 1e-7 for a, b in zip(q, exact.charges()))
    cold_launches, cold_its, cold_q = solve(None)
    assert cold_its.min() > 10 and cold_launches >= cold_its.max() - 1     # (the setup counts as one)
    if len(parts) > 1:
        launches, its, q = solve([None] + hist[1:])
        assert tuple(its[0]) == tuple(cold_its[0]) and its[1:].max() == 1
        assert np.array_equal(q[0], cold_q[0])
