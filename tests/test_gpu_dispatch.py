"""Both sides of the size rules that choose between kernel variants, against the oracle."""
import numpy as np
import pytest

from conftest import compare_tree, rel_l2

pytestmark = pytest.mark.gpu


# census items per wave (2^20 sources), lanes per node of the topology search (16,384 internal
# nodes), blocks of 1,024 and 4,096 positions, one-source leaves down to level 15, a lone leaf
@pytest.mark.parametrize("n,leaf", [(1, 1), (2, 1), (64, 1), (1023, 1), (1025, 3), (4097, 1), (20000, 1),
                                    (1 << 20, 32), ((1 << 20) + 1, 512), ((1 << 20) + 4095, 24)])
def test_topology_variants(pkg, oracle, wl, n, leaf):
    xs, ys, vs, *_ = wl.mixed_plummer_potential(n, seed=n % 97)
    ctx = pkg.Context(pot_order=6, pot_leaf=leaf)
    ctx.potential(0.5, xs, ys, vs, xs[:1], ys[:1])
    compare_tree(ctx.tree(), oracle.Tree(xs, ys, vs, leaf, 6))
    ctx.close()


# the upward pass above the leaves: every level in the chained launch (at most 4,096 internal
# nodes), the lower ones level by level beyond; one order per lane-group width
@pytest.mark.parametrize("n,leaf,order", [(3, 1, 6), (5000, 1, 16), (60000, 16, 20), (200000, 12, 16),
                                          (300000, 8, 32), (100000, 1, 9)])
def test_upward_variants(pkg, oracle, wl, n, leaf, order):
    xs, ys, vs, *_ = wl.mixed_plummer_potential(n, seed=order)
    ctx = pkg.Context(force_order=order, force_leaf=leaf)
    ctx.force(0.5, xs, ys, vs, np.array([0.4]), np.array([0.4]), np.array([1.0 / 512]))
    compare_tree(ctx.tree(), oracle.Tree(xs, ys, vs, leaf, order))
    ctx.close()


# leaf sums: every order's split of the values over the lanes (halves of odd and even counts); leaves
# of 1 to 64 points and of several 64s
@pytest.mark.parametrize("order", [6, 8, 9, 10, 12, 14, 16, 20, 24, 32])
@pytest.mark.parametrize("n,leaf", [(1, 1), (64, 64), (65, 65), (129, 200), (3001, 64), (3001, 257)])
def test_leaf_orders(pkg, oracle, wl, n, leaf, order):
    xs, ys, vs, *_ = wl.mixed_plummer_potential(n, seed=n + order)
    ctx = pkg.Context(force_order=order, force_leaf=leaf)
    ctx.force(0.5, xs, ys, vs, np.array([0.4]), np.array([0.4]), np.array([1.0 / 512]))
    compare_tree(ctx.tree(), oracle.Tree(xs, ys, vs, leaf, order))
    ctx.close()


# one-workgroup sorts with 1, 2, 4, 8, 12, 16 keys per thread, one-launch passes with 1,024 threads a
# tile (up to 256 tiles of 5,120 keys) and 256 beyond; many equal keys, so stability shows
@pytest.mark.parametrize("n", [1, 1024, 1025, 2048, 2049, 4096, 4097, 8192, 8193, 12288, 12289, 16384, 16385, 40961,
                               256 * 5120, 256 * 5120 + 1])
def test_sort_variants(pkg, oracle, wl, n):
    st = wl.Stream(n)
    x, y = np.floor(st.uniform(n) * 50) / 50, np.floor(st.uniform(n) * 40) / 40
    ctx = pkg.Context()
    box, keys, perm = ctx.empty(4), ctx.empty(n, np.uint32), ctx.empty(n, np.uint32)
    ctx.morton_sort_device(ctx.to_device(x), ctx.to_device(y), box, keys, perm)
    ctx.synchronize()
    obox = oracle.bbox(x, y)
    operm, oks = oracle.sort(oracle.keys(x, y, obox))
    assert np.array_equal(box.numpy()[:3], obox)
    assert np.array_equal(keys.numpy(), oks) and np.array_equal(perm.numpy(), operm)
    ctx.close()


# one-launch passes with 5, 8 and 15 keys per thread: whole tiles, one key more or less, the largest
# of each; few distinct keys, and keys in their order and in reverse
@pytest.mark.parametrize("n", [3 * 5120, 4 * 5120 + 1, 256 * 5120 + 8192, 257 * 8192 - 1, 1 << 22, (1 << 22) + 1,
                               274 * 15360])
def test_sort_tiles(pkg, oracle, wl, n):
    st = wl.Stream(n)
    t = np.arange(n) / n
    for x, y in [(np.floor(st.uniform(n) * 3) / 3, np.floor(st.uniform(n) * 4) / 4), (t, t), (1 - t, 0 * t)]:
        ctx = pkg.Context()
        box, keys, perm = ctx.empty(4), ctx.empty(n, np.uint32), ctx.empty(n, np.uint32)
        ctx.morton_sort_device(ctx.to_device(x), ctx.to_device(y), box, keys, perm)
        ctx.synchronize()
        operm, oks = oracle.sort(oracle.keys(x, y, oracle.bbox(x, y)))
        assert np.array_equal(keys.numpy(), oks) and np.array_equal(perm.numpy(), operm)
        ctx.close()


# FP64 potential: 8, 16, 32, 64 targets per wave, whatever the wave the same bits; leaves of one
# and of several source tiles, full and ragged; 1 to 64 active lanes a leaf
@pytest.mark.parametrize("m", [1, 7, 8192, 8193, 49152, 49153, 98304, 98305])
@pytest.mark.parametrize("order,leaf", [(9, 33), (12, 500)])
def test_fp64_targets_per_wave(pkg, oracle, wl, m, order, leaf):
    xs, ys, vs, *_ = wl.mixed_plummer_potential(30011, seed=m % 89)
    st = wl.Stream(m)
    xt, yt = st.uniform(m, -0.2, 1.2), st.uniform(m, -0.2, 1.2)
    ctx = pkg.Context(pot_order=order, pot_leaf=leaf, counters=True)
    out = ctx.potential(0.5, xs, ys, vs, xt, yt)
    cnt = ctx.stats()["counters"]
    idx = np.sort(np.random.default_rng(m).choice(m, min(m, 2000), replace=False))
    ot = oracle.Tree(xs, ys, vs, leaf, order)
    ref, rc = ot.potential(0.5, xt[idx], yt[idx])
    assert rel_l2(out[idx], ref) <= 1e-12
    if len(idx) == m:
        assert (cnt["p2p"], cnt["e2p"]) == (rc[0], rc[1])
    for part in (idx, idx[:9], idx[-1:]):
        assert np.array_equal(ctx.potential_resident(0.5, xt[part], yt[part]), out[part])
    ctx.close()


def test_fp64_potential_nonfinite_and_huge(pkg):
    # log64 takes finite positive arguments; what overflows a squared distance is NaN, as log is there
    ctx = pkg.Context()
    xs, ys, vs = np.array([0.0, 1.0]), np.array([0.0, 1.0]), np.array([1.0, -2.0])
    x = np.array([0.5, 1e200, np.inf, np.nan, -1e160, 0.0])
    y = np.array([0.5, 0.0, 0.0, 0.0, 1e160, 0.0])
    d = [ctx.to_device(a) for a in (xs, ys, vs, x, y)]
    out = ctx.empty(len(x))
    ctx.potential(0.0, *d, out=out, device=True)
    ctx.synchronize()
    o = out.numpy()
    assert np.isnan(o[[1, 2, 3, 4]]).all() and np.isfinite(o[[0, 5]]).all()
    eps = 10 * np.finfo(float).eps
    want = [sum(v * 0.5 * np.log((a - s) ** 2 + (b - t) ** 2 + eps) for s, t, v in zip(xs, ys, vs))
            for a, b in zip(x[[0, 5]], y[[0, 5]])]
    assert np.allclose(o[[0, 5]], want, rtol=1e-14, atol=1e-15)
    ctx.close()


# force at targets: the same rule; a target's result is the same alone and among others
@pytest.mark.parametrize("m", [1, 9, 8192, 8193, 49153, 98305])
@pytest.mark.parametrize("precision", [0, 1])
def test_force_targets_per_wave(pkg, oracle, wl, m, precision):
    xs, ys, vs, *_ = wl.gaussian4_force(20011, seed=m % 83)
    st = wl.Stream(m)
    xt, yt = st.uniform(m), st.uniform(m)
    ctx = pkg.Context(precision=precision, force_order=12, force_leaf=70)
    fx, fy = ctx.force_targets(0.5, xs, ys, vs, xt, yt)
    idx = np.sort(np.random.default_rng(m).choice(m, min(m, 500), replace=False))
    rx, ry, _ = oracle.force_targets(0.5, xs, ys, vs, xt[idx], yt[idx], order=12, leafcap=70)
    tol = 1e-5 if precision else 1e-12
    assert rel_l2(fx[idx], rx) <= tol and rel_l2(fy[idx], ry) <= tol
    gx, gy = ctx.force_targets(0.5, xs, ys, vs, xt[idx[:17]], yt[idx[:17]])
    assert np.array_equal(gx, fx[idx[:17]]) and np.array_equal(gy, fy[idx[:17]])
    ctx.close()


def test_fp64_force_on_fp32_tree(pkg, wl):
    # a tree built for FP32 keeps no k a_k of its own: an FP64 evaluation of it adds them
    xs, ys, vs, x0s, y0s, hs = wl.gaussian4_force(30000, seed=5, nbx=4, h=1.0 / 128)
    ctx = pkg.Context(precision=pkg.FP64, force_order=10, force_leaf=64)
    want = ctx.force(0.5, xs, ys, vs, x0s, y0s, hs)
    ctx.set(pkg.OPT_PRECISION, pkg.FP32)
    ctx.force(0.5, xs, ys, vs, x0s, y0s, hs)
    ctx.set(pkg.OPT_PRECISION, pkg.FP64)
    for _ in range(2):
        got = ctx.force_resident(0.5, x0s, y0s, hs)
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
    ctx.close()


# float arrays are converted on the GPU: packed (one transfer), array by array, and with targets
# uploaded beside the build; forces in one piece and in ranges
@pytest.mark.parametrize("n,m", [(5, 3), (1001, 777), (1 << 20, 70001), (100001, 1 << 20)])
def test_float_arrays_equal_double_arrays(pkg, wl, n, m):
    st = wl.Stream(n + m)
    a = [st.uniform(n).astype(np.float32), st.uniform(n).astype(np.float32), st.uniform(n, -1, 1).astype(np.float32),
         st.uniform(m).astype(np.float32), st.uniform(m).astype(np.float32)]
    out = pkg.treecode_potential_float(0.5, *a)
    ctx = pkg.Context(precision=pkg.FP32)
    ref = ctx.potential(float(np.float32(0.5)), *[v.astype(np.float64) for v in a])
    assert out.dtype == np.float32 and np.array_equal(out, ref.astype(np.float32))
    ctx.close()


@pytest.mark.parametrize("nb", [1, 33, 2050])
def test_float_forces_equal_double_forces(pkg, wl, nb):
    xs, ys, vs, x0s, y0s, hs = wl.gaussian4_force(20000, seed=nb)
    a = [v.astype(np.float32) for v in (xs, ys, vs, x0s[:nb], y0s[:nb], hs[:nb])]
    fx, fy = pkg.treecode_force_mrag_float(0.5, *a)
    ctx = pkg.Context(precision=pkg.FP32)
    rx, ry = ctx.force(0.5, *[v.astype(np.float64) for v in a])
    assert np.array_equal(fx, rx.astype(np.float32)) and np.array_equal(fy, ry.astype(np.float32))
    ctx.close()


# topology by the sorting workgroup (up to 1,024 internal nodes by the bound) and by its own kernels;
# a tree queued at its node bound and one that waits for its census; sources and targets sorted
# together (both small, both middling) and apart
@pytest.mark.parametrize("n,m,leaf", [(1, 1, 1), (2, 3, 1), (70, 1000, 1), (900, 16384, 64), (16384, 1, 200),
                                      (16384, 16385, 200), (16385, 16384, 200), (12000, 9000, 8), (20000, 20001, 2),
                                      (20000, 30000, 300), (600000, 448576, 512), (600000, 448577, 512)])
def test_build_queueing_variants(pkg, oracle, wl, n, m, leaf):
    xs, ys, vs, *_ = wl.mixed_plummer_potential(n, seed=leaf)
    st = wl.Stream(m)
    xt, yt = st.uniform(m), st.uniform(m)
    ctx = pkg.Context(pot_order=8, pot_leaf=leaf)
    ot = oracle.Tree(xs, ys, vs, leaf, 8)
    idx = np.sort(np.random.default_rng(m).choice(m, min(m, 300), replace=False))
    ref, _ = ot.potential(0.5, xt[idx], yt[idx])
    for _ in range(2):
        out = ctx.potential(0.5, xs, ys, vs, xt, yt)
        assert rel_l2(out[idx], ref) <= 1e-12
    compare_tree(ctx.tree(), ot)
    # non-finite coordinates are reported, and the context stays usable
    for bad in (0, n - 1):
        b = xs.copy()
        b[bad] = np.nan
        with pytest.raises(pkg.TreecodeError):
            ctx.potential(0.5, b, ys, vs, xt, yt)
    b = xt.copy()
    b[-1] = np.inf
    with pytest.raises(pkg.TreecodeError):
        ctx.potential(0.5, xs, ys, vs, b, yt)
    assert np.array_equal(ctx.potential(0.5, xs, ys, vs, xt, yt), out)
    ctx.close()
