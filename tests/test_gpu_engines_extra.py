"""The `hip_block` and `hip_ah` engines (GPU counterparts of the reference's
`block` and `ah` CPU engines, nbody/nbody_engine_block.cpp:14-126 and
nbody/nbody_engine_ah.cpp:16-160) against the oracle's restatements, bit for
bit, through the C ABI and through the engine interface."""
import ctypes as C

import numpy as np
import pytest

import oracle_lib
from hip_capi import Ctx
from nbody_amd import native, nbody_create_engine, nbody_create_solver, nbody_data

pytestmark = pytest.mark.gpu

NBH_FP64_BLOCK = 3


@pytest.fixture(scope="module")
def ctx():
    c = Ctx(0)
    yield c
    c.close()


def _data(kind, n, seed):
    d = nbody_data()
    d.set_quiet(True)
    d.generate(kind, n, seed)
    return d


def _state(kind, n, seed):
    return oracle_lib.state_from_data(_data(kind, n, seed))


# (up to 4096 bodies on 256 CUs the work-group size is checked and chooses nothing; the
# form that uses it is tested in test_gpu_direct.py)
@pytest.mark.parametrize("n,bs", [(1, 0), (64, 64), (100, 128), (1000, 256), (1536, 1024), (4096, 0)])
def test_block_bit_exact(ctx, n, bs):
    y, m = _state("plummer", n, 21 + n)
    dy, dm, df = ctx.put(y), ctx.put(m), ctx.alloc(6 * n)
    native.check(ctx.lib.nbh_fcompute_direct(ctx.h, dy.ptr, dm.ptr, df.ptr, n, NBH_FP64_BLOCK, bs), "block")
    assert np.array_equal(df.read(), oracle_lib.fcompute_block(y, m))


def test_block_out_of_range_operands(ctx):
    """Coincident bodies, a clamped pair, a zero mass and a coordinate beyond
    1e6 take the general division and root; still the oracle's bits."""
    pos = np.array([[0, 0, 0], [0, 0, 0], [1e-5, 0, 0], [2e6, 1, 1], [3, 4, 5]], dtype=np.float64)
    m = np.array([1.0, 2.0, 0.0, 3.0, 4.0])
    y = np.concatenate([pos[:, 0], pos[:, 1], pos[:, 2], np.arange(15, dtype=np.float64)])
    dy, dm, df = ctx.put(y), ctx.put(m), ctx.alloc(30)
    native.check(ctx.lib.nbh_fcompute_direct(ctx.h, dy.ptr, dm.ptr, df.ptr, 5, NBH_FP64_BLOCK, 64), "block")
    assert np.array_equal(df.read(), oracle_lib.fcompute_block(y, m))


def test_block_engine_reference_test():
    """test/engine/test_nbody_engine.cpp:1180-1187: the engine on
    make_universe(64) against `simple`, |f - f0| <= 1e-13, and the oracle's
    block bits."""
    d = nbody_data()
    d.set_quiet(True)
    d.make_universe(64, 100, 100, 100)
    y, m = oracle_lib.state_from_data(d)
    e = nbody_create_engine({"engine": "hip_block"})
    assert e is not None and e.init(d)
    assert e.type_name() == "nbody_engine_hip_block"
    f = e.create_buffer(8 * len(y))
    e.fcompute(0.0, e.get_y(), f)
    out = e.read_buffer(f)
    assert np.max(np.abs(out - oracle_lib.fcompute_simple(y, m))) <= 1e-13
    assert np.array_equal(out, oracle_lib.fcompute_block(y, m))
    e.free_buffer(f)
    e.destroy()


def test_block_rk4_trajectory_equals_oracle():
    d1, d2 = _data("ball", 512, 3), _data("ball", 512, 3)
    eh = nbody_create_engine({"engine": "hip_block"})
    eo = oracle_lib.block_engine(0)
    assert eh.init(d1) and eo.init(d2)
    for e in (eh, eo):
        s = nbody_create_solver({"solver": "rk4", "max_step": 1e-3})
        s.set_engine(e)
        for _ in range(10):
            s.advise(1e-3)
        s.destroy()
    assert np.array_equal(eh.read_buffer(eh.get_y()), eo.read_buffer(eo.get_y()))
    eh.destroy()
    eo.destroy()


def _ah_lists(ctx, ah, n):
    total = C.c_size_t()
    native.check(ctx.lib.nbh_ah_lists(ctx.h, ah, C.byref(total), None, None, None), "lists")
    offs = np.empty(n + 1, np.uint64)
    lst = np.empty(max(1, total.value), np.uint32)
    univ = np.empty(3 * n)
    native.check(ctx.lib.nbh_ah_lists(ctx.h, ah, C.byref(total), offs.ctypes.data_as(C.c_void_p),
                                      lst.ctypes.data_as(C.c_void_p), univ.ctypes.data_as(C.c_void_p)), "lists")
    return offs, lst[:total.value], univ.reshape(3, n).T


@pytest.mark.parametrize("kind,n,dist,force", [("plummer", 1000, 0.3, 2e-6), ("ball", 4097, 0.2, 1e-5),
                                                ("plummer", 256, 1e9, 0.0), ("cube", 300, 0.0, np.inf)])
def test_ah_full_and_sparse_bit_exact(ctx, kind, n, dist, force):
    y, m = _state(kind, n, 31)
    ah = C.c_void_p()
    native.check(ctx.lib.nbh_ah_create(ctx.h, n, C.byref(ah)), "ah create")
    try:
        dy, dm, df = ctx.put(y), ctx.put(m), ctx.alloc(6 * n)
        # a sparse pass before any full pass is refused
        assert ctx.lib.nbh_ah_fcompute_sparse(ctx.h, ah, dy.ptr, dm.ptr, df.ptr) == 1
        native.check(ctx.lib.nbh_ah_fcompute_full(ctx.h, ah, dy.ptr, dm.ptr, df.ptr, dist, force), "full")
        o = oracle_lib.AH(n, dist, force)
        f0 = o.full(y, m)
        assert np.array_equal(df.read(), f0)
        offs, lst, univ = _ah_lists(ctx, ah, n)
        ooffs, olst, ouniv = o.lists()
        assert np.array_equal(offs, ooffs) and np.array_equal(lst, olst)
        assert np.array_equal(univ, ouniv)
        # sparse pass at moved positions
        rng = np.random.default_rng(n)
        y2 = y.copy()
        y2[:3 * n] += rng.normal(0, 1e-3, 3 * n)
        dy.write(y2)
        native.check(ctx.lib.nbh_ah_fcompute_sparse(ctx.h, ah, dy.ptr, dm.ptr, df.ptr), "sparse")
        assert np.array_equal(df.read(), o.sparse(y2, m))
    finally:
        native.check(ctx.lib.nbh_ah_destroy(ah), "ah destroy")


def test_ah_lists_grow(ctx):
    """A second full pass with more neighbours than the first regrows the lists."""
    n = 2048
    y, m = _state("plummer", n, 5)
    ah = C.c_void_p()
    native.check(ctx.lib.nbh_ah_create(ctx.h, n, C.byref(ah)), "ah create")
    try:
        dy, dm, df = ctx.put(y), ctx.put(m), ctx.alloc(6 * n)
        totals = []
        for dist in (0.05, 0.5, 0.1):
            native.check(ctx.lib.nbh_ah_fcompute_full(ctx.h, ah, dy.ptr, dm.ptr, df.ptr, dist, 1e9), "full")
            o = oracle_lib.AH(n, dist, 1e9)
            o.full(y, m)
            offs, lst, _ = _ah_lists(ctx, ah, n)
            ooffs, olst, _ = o.lists()
            assert np.array_equal(offs, ooffs) and np.array_equal(lst, olst)
            totals.append(len(lst))
        assert totals[0] < totals[2] < totals[1]
    finally:
        native.check(ctx.lib.nbh_ah_destroy(ah), "ah destroy")


def test_ah_engine_reference_test():
    """test/engine/test_nbody_engine.cpp:1169-1178: `ah` with rate 5, max_dist 7,
    min_force 1e-6 on make_universe(64) at step 0, |f - f0| <= 1e-13 against
    `simple` (a full recompute: the simple sum itself)."""
    d = nbody_data()
    d.set_quiet(True)
    d.make_universe(64, 100, 100, 100)
    y, m = oracle_lib.state_from_data(d)
    e = nbody_create_engine({"engine": "hip_ah", "full_recompute_rate": 5, "max_dist": 7, "min_force": 1e-6})
    assert e is not None and e.init(d)
    f = e.create_buffer(8 * len(y))
    e.set_step(0)
    e.fcompute(0.0, e.get_y(), f)
    out = e.read_buffer(f)
    f0 = oracle_lib.fcompute_simple(y, m)
    assert np.max(np.abs(out - f0)) <= 1e-13
    assert np.array_equal(out, f0)
    e.free_buffer(f)
    e.destroy()


@pytest.mark.parametrize("solver", ["rk4", "euler"])
def test_ah_trajectory_equals_oracle(solver):
    """Full recomputes every 4 steps, sparse passes in between: the trajectory
    and the neighbour lists equal the oracle engine's bit for bit."""
    n = 1024
    d1, d2 = _data("plummer", n, 8), _data("plummer", n, 8)
    keys = {"full_recompute_rate": 4, "max_dist": 0.25, "min_force": 1e-6}
    eh = nbody_create_engine({"engine": "hip_ah", **keys})
    eo = oracle_lib.ah_engine(4, 0.25, 1e-6)
    assert eh.init(d1) and eo.init(d2)
    for e in (eh, eo):
        s = nbody_create_solver({"solver": solver, "max_step": 1e-3})
        s.set_engine(e)
        for _ in range(10):
            s.advise(1e-3)
        s.destroy()
    assert eh.get_compute_count() == eo.get_compute_count()
    assert np.array_equal(eh.read_buffer(eh.get_y()), eo.read_buffer(eo.get_y()))
    ctx = native.hip_lib()
    total = C.c_size_t()
    native.check(ctx.nbh_ah_lists(eh.hip_context(), eh.hip_neighbours(), C.byref(total), None, None, None), "lists")
    ooffs, olst = oracle_lib.ah_engine_lists(eo, n)
    assert total.value == len(olst) > 0
    eh.destroy()
    eo.destroy()
