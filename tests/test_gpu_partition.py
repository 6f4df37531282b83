"""QEq after swr_set_batch regroups the atoms between the H build and the
solve.  H does not depend on the partition, so the charges, solutions and
iteration counts are those of a system that had the final partition from the
start, bit for bit, whichever of the three FP64 forms (one launch for the
solve, one per iteration, the general one) either partition takes."""
import ctypes as C

import numpy as np
import pytest

from sw_reaxff_amd import batch, systems

from .test_zz_no_alloc import D2H, H2D, _hip, _ok

pytestmark = pytest.mark.gpu


def waters(m, seed):
    s = systems.water_box(m, seed=seed)
    return systems.System(x=s.x, v=s.v, type=s.type, tag=s.tag, elements=s.elements, lo=s.x.min(0) - 12.0,
                          hi=s.x.max(0) + 12.0, periodic=False)


def loaded(gpu_lib, ffield, P, groups, mixed=0):
    """A system of the packed atoms with H built under the partition `groups`
    (numbers of consecutive packed systems that make one system each)."""
    h = gpu_lib.System(ffield, batch.ELEMENTS, tol=1e-6, qeq_mixed=mixed)
    h.set_atoms(P.n, P.x, P.type, P.tag, owner=P.owner, img=P.img)
    regroup(gpu_lib, h, P, groups)
    h.build_neighbors(batch.CUTGHOST)
    h.call("qeq_init_matvec")
    return h


def regroup(gpu_lib, h, P, groups):
    o = np.ascontiguousarray(P.row_off[np.concatenate([[0], np.cumsum(groups)])], dtype=np.int32)
    assert o[-1] == P.n
    gpu_lib.check(h.L.swr_set_batch(h.h, len(groups), o.ctypes.data_as(C.POINTER(C.c_int))), "swr_set_batch")


def solved(h):
    its = h.qeq_cg()
    h.call("calculate_q")
    h.sync()
    return its, h.get("sys_iters"), h.get("s"), h.get("t"), h.get("q")


SIZES = {"tiny": [1, 7, 21, 20], "small": [30, 100, 7, 450], "general": [700, 700, 400], "large": [1100, 30, 1200]}


@pytest.mark.parametrize("mixed", [0, 1])
@pytest.mark.parametrize("sizes,before,after", [
    ("tiny", [1, 1, 1, 1], [4]),            # one launch a solve -> one an iteration
    ("tiny", [4], [1, 1, 1, 1]),
    ("tiny", [1, 1, 1, 1], [2, 1, 1]),      # fewer systems, more, other ones
    ("small", [1, 1, 1, 1], [2, 2]),
    ("small", [2, 2], [1, 1, 1, 1]),
    ("small", [1, 3], [3, 1]),
    ("general", [1, 1, 1], [3]),            # small -> general (5,400 rows)
    ("general", [3], [1, 1, 1]),
    ("general", [1, 1, 1], [2, 1]),
    ("large", [3], [1, 1, 1]),              # general either way
    ("large", [1, 1, 1], [2, 1]),
])
def test_gpu_regrouped_between_build_and_solve(gpu_lib, ffield, sizes, before, after, mixed):
    P = batch.pack([waters(m, seed=m) for m in SIZES[sizes]])
    ref = loaded(gpu_lib, ffield, P, after, mixed)
    h = loaded(gpu_lib, ffield, P, before, mixed)
    regroup(gpu_lib, h, P, after)
    for _ in range(2):
        want, got = solved(ref), solved(h)
        assert got[0] == want[0] and want[0][0] > 2
        for g, w in zip(got[1:], want[1:]):
            assert np.array_equal(g, w)
        for k in (ref, h):                  # and once more with H built under the new one
            k.call("qeq_init_matvec")


@pytest.mark.parametrize("sizes,before", [("tiny", [1, 1, 1, 1]), ("tiny", [2, 2]), ("small", [2, 2]),
                                          ("general", [1, 1, 1]), ("large", [1, 1, 1])])
def test_gpu_noalloc_after_regrouping(gpu_lib, ffield, sizes, before):
    """The no-allocation solve of the systems merged into one."""
    hip = _hip()
    P = batch.pack([waters(m, seed=m) for m in SIZES[sizes]])
    one = [len(SIZES[sizes])]
    ref = loaded(gpu_lib, ffield, P, one)
    h = loaded(gpu_lib, ffield, P, before)
    regroup(gpu_lib, h, P, one)
    h.sync()
    b = np.ascontiguousarray(np.stack([h.get("b_s"), h.get("b_t")], axis=1))
    x = np.ascontiguousarray(np.stack([h.get("s"), h.get("t")], axis=1))
    want = solved(ref)
    db, dx = C.c_void_p(), C.c_void_p()
    _ok(hip.hipMalloc(C.byref(db), b.nbytes), "hipMalloc b")
    _ok(hip.hipMalloc(C.byref(dx), x.nbytes), "hipMalloc x")
    try:
        _ok(hip.hipMemcpy(db, b.ctypes.data, b.nbytes, H2D), "copy b")
        _ok(hip.hipMemcpy(dx, x.ctypes.data, x.nbytes, H2D), "copy x")
        i, j = C.c_int(0), C.c_int(0)
        gpu_lib.check(h.L.swr_qeq_cg_noalloc(h.h, db, dx, C.byref(i), C.byref(j)), "swr_qeq_cg_noalloc")
        _ok(hip.hipMemcpy(x.ctypes.data, dx, x.nbytes, D2H), "copy x back")
    finally:
        hip.hipFree(db)
        hip.hipFree(dx)
    assert (i.value, j.value) == want[0]
    assert np.array_equal(x[:, 0], want[2]) and np.array_equal(x[:, 1], want[3])
    got = solved(h)                          # the allocating solve afterwards
    assert got[0] == want[0] and np.array_equal(got[4], want[4])


def test_gpu_autotune_after_regrouping(gpu_lib, ffield):
    P = batch.pack([waters(m, seed=m) for m in SIZES["general"]])
    for before, after in (([1, 1, 1], [3]), ([3], [1, 1, 1])):
        want = solved(loaded(gpu_lib, ffield, P, after))
        h = loaded(gpu_lib, ffield, P, before)
        regroup(gpu_lib, h, P, after)
        rep = h.autotune(reps=2)
        assert all(v > 0 for v in rep["spmv_fp64"]["us"].values())
        h.set_shape("spmv_fp64", "T512G8U4")
        got = solved(h)
        assert got[0] == want[0] and np.array_equal(got[4], want[4])


def test_gpu_solve_needs_the_h_of_its_atoms(gpu_lib, ffield):
    """After swr_set_atoms with another number of atoms the old H has no rows
    for them: every solve says so until swr_qeq_init_matvec."""
    P = batch.pack([waters(30, seed=1)])
    Q = batch.pack([waters(45, seed=2)])
    want = solved(loaded(gpu_lib, ffield, Q, [1]))
    h = loaded(gpu_lib, ffield, P, [1])
    h.set_atoms(Q.n, Q.x, Q.type, Q.tag, owner=Q.owner, img=Q.img)
    dev = h.L.swr_device_ptr(h.h, b"x")
    for call in (lambda: h.qeq_cg(),
                 lambda: gpu_lib.check(h.L.swr_qeq_cg_noalloc(h.h, dev, dev, None, None), "swr_qeq_cg_noalloc")):
        with pytest.raises(gpu_lib.SwrError) as e:
            call()
        assert e.value.code == 6                 # SWR_ERR_STATE
    assert "spmv_fp64" not in h.autotune(reps=1)
    gpu_lib.check(h.L.swr_new_atoms(h.h), "swr_new_atoms")
    h.build_neighbors(batch.CUTGHOST)
    h.call("qeq_init_matvec")
    got = solved(h)
    assert got[0] == want[0] and np.array_equal(got[4], want[4])


def test_gpu_panel_lists_are_read_of_the_current_h_only(gpu_lib, ffield):
    """A small system's column lists are made when they are asked for; between
    swr_set_atoms with another number of atoms and the next H there are none
    (more rows than the arrays held, and fewer)."""
    names = ("panel_count", "panel_columns", "H_jloc")
    P = batch.pack([waters(30, seed=1)])
    h = loaded(gpu_lib, ffield, P, [1])
    for m in (300, 12):
        Q = batch.pack([waters(m, seed=m)])
        h.set_atoms(Q.n, Q.x, Q.type, Q.tag, owner=Q.owner, img=Q.img)
        assert all(h.get(k).size == 0 for k in names)
        assert not any(h.L.swr_device_ptr(h.h, k.encode()) for k in names)
        h.build_neighbors(batch.CUTGHOST)
        h.call("qeq_init_matvec")
        f, nn, jl, loc = h.get("H_firstnbr"), h.get("H_numnbrs"), h.get("H_jlist"), h.get("H_jloc")
        pb, cnt, col = h.get("panel_begin"), h.get("panel_count"), h.get("panel_columns")
        rows = h.get("panel_rows")
        assert cnt.size == -(-Q.n // 64) and pb[-1] == Q.n
        for p in range(cnt.size):
            for i in rows[pb[p]:pb[p + 1]]:
                e = slice(f[i], f[i] + nn[i])
                assert np.array_equal(col[p * gpu_lib.PANEL_MAXC + loc[e]], jl[e])


def test_gpu_autotune_times_the_small_solve(gpu_lib, ffield):
    """For small systems the FP64 family's shapes are those of the one-launch
    steps, which use no column lists: timing them makes none (13 MB here)."""
    hip = _hip()
    hip.hipMemGetInfo.argtypes = [C.POINTER(C.c_size_t)] * 2

    def free():
        a, b = C.c_size_t(0), C.c_size_t(0)
        _ok(hip.hipDeviceSynchronize(), "synchronize")
        _ok(hip.hipMemGetInfo(C.byref(a), C.byref(b)), "hipMemGetInfo")
        return a.value

    P = batch.pack([waters(1, seed=k) for k in range(960)] + [waters(22, seed=2000)])
    h = loaded(gpu_lib, ffield, P, [1] * 961)
    solved(h)
    lists = 4 * gpu_lib.PANEL_MAXC * 962
    before = free()
    rep = h.autotune(reps=2)
    assert before - free() < lists // 2
    assert set(rep["spmv_fp64"]["us"]) == {"T512G8U4", "T512G8U2", "T256G8U4", "T256G4U4"}
    h.get("panel_count")
    assert before - free() >= lists // 2       # (the probe sees the lists when they are made)
