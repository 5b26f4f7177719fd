"""The level-synchronous driver's neighbour walks against the oracle on data
whose coordinates sit on the edges of the eps cells (one float to either side,
exactly on them, and half a cell away), where the cell rule and the distance
disagree; whole results are compared, with per-tree traces."""

import sys

import numpy as np
import pytest

from gpu_inscy_amd import _lib, datagen
from gpu_inscy_amd import inscy as INSCY
from oracle import oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    _lib.lib()


def edge_data(seed, n, d, eps):
    """Points of d-dimensional clumps on a lattice of half eps cells, moved by at
    most one float in a third of the coordinates."""
    rng = np.random.default_rng(seed)
    C = int(np.ceil(1.0 / np.float64(np.float32(eps))))
    centre = rng.integers(2, 2 * C - 2, size=(max(2, n // 60), d))
    at = centre[rng.integers(0, len(centre), n)] + rng.integers(-2, 3, size=(n, d))
    at = np.where(rng.random((n, d)) < 0.15, rng.integers(0, 2 * C + 1, size=(n, d)), at)
    X = np.clip(at.astype(np.float64) / (2 * C), 0.0, 1.0).astype(np.float32)
    step = rng.random((n, d))
    X = np.where(step < 1 / 6, np.nextafter(X, np.float32(0)), X)
    X = np.where(step > 5 / 6, np.nextafter(X, np.float32(1)), X)
    return np.clip(X, 0.0, 1.0).astype(np.float32)


# eps whose reciprocal is whole (cells of width eps up to rounding) and not
# (cells narrower than eps: neighbours by distance in cells two apart)
@pytest.mark.parametrize("rect", [True, False])
@pytest.mark.parametrize("n,d,eps,num_obj", [(300, 4, 0.05, 3), (1201, 5, 0.05, 4), (1300, 6, 0.03, 3),
                                             (700, 7, 0.125, 5), (257, 9, 0.11, 4)])
def test_walks_on_cell_edges_match_oracle(n, d, eps, num_obj, rect):
    print("cell edges", n, d, eps, num_obj, rect, flush=True)
    sys.stdout.flush()
    X = edge_data(n + d, n, d, eps)
    args = (eps, 1.0, num_obj, max(4, n // 40), 1.0, 4, rect, 0)
    ref = O.run_ref(X, *args[:7], 0, trace=True)
    _lib.debug_trace(True)
    try:
        got = INSCY.run(X, *args, mode=_lib.MODE_BATCHED)
        trace = _lib.debug_trace_rows()
    finally:
        _lib.debug_trace(False)
    assert got.subspaces == ref.subspaces
    for s, a, b in zip(ref.subspaces, ref.labels, got.labels):
        assert np.array_equal(O.canonical(a), b), f"labels differ in subspace {s}"
    assert np.array_equal(trace, ref.trace)
    assert max(len(s) for s in got.subspaces) >= 3


# masks whose children are counted by one walk: up to 3, 7, 15 and 31 children
# (the widths of the walk; test_wide_dimensions_match_oracle has more than 64),
# with points of clumps that stay dense over many dimensions (walks of 1 to 4)
@pytest.mark.parametrize("n,d,eps,dims,rect", [(260, 5, 0.04, 5, True), (260, 5, 0.04, 5, False),
                                               (350, 9, 0.04, 5, True), (350, 9, 0.04, 5, False),
                                               (300, 17, 0.02, 4, True), (300, 17, 0.02, 4, False),
                                               (301, 33, 0.02, 4, True)])
def test_walks_serving_many_children_match_oracle(n, d, eps, dims, rect):
    print("children", n, d, eps, dims, rect, flush=True)
    rng = np.random.default_rng(n * d)
    X = rng.random((n, d)).astype(np.float32)
    for c in range(3):
        rows = np.arange(c * n // 4, (c + 1) * n // 4)[:, None]
        at = np.sort(rng.choice(d, dims, replace=False)) if c else np.r_[0:dims - 1, d - 1]
        size = (c + 1) * n // 4 - c * n // 4
        X[rows, at] = (rng.uniform(0.2, 0.8, dims) + 0.4 * eps * rng.standard_normal((size, dims))).astype(np.float32)
    X = np.clip(X, 0.0, 1.0)
    args = (eps, 1.0, 4, n // 6, 1.0, 4, rect, 0)
    ref = O.run_ref(X, *args[:7], 0, trace=True)
    _lib.debug_trace(True)
    try:
        got = INSCY.run(X, *args, mode=_lib.MODE_BATCHED)
        trace = _lib.debug_trace_rows()
    finally:
        _lib.debug_trace(False)
    assert got.subspaces == ref.subspaces
    for s, a, b in zip(ref.subspaces, ref.labels, got.labels):
        assert np.array_equal(O.canonical(a), b), f"labels differ in subspace {s}"
    assert np.array_equal(trace, ref.trace)
    assert max(len(s) for s in got.subspaces) >= dims - 1


def groups(n, per):
    """n points in tight groups of `per` on a grid, and each point's group, line and
    column: n / per groups in the pair of columns (their number decides whether
    its first parents fit the LDS), the square root of that in either one."""
    rng = np.random.default_rng(n + per)
    k = n // per
    g = int(np.ceil(np.sqrt(k)))
    at = rng.permutation(np.minimum(np.arange(n) // per, k - 1))
    X = np.stack([at // g, at % g], 1) + 0.4 + rng.uniform(0, 0.11, (n, 2))
    return (X / g).astype(np.float32), 0.25 / g, (at // g, at % g, at)


# k_b_sample's rules at 39,936 points (ids in LDS up to there) and four times
# that (global parents above); groups of 3 leave more first parents than fit
# from 119,808 points on
@pytest.mark.parametrize("n,per", [(75, 3), (1025, 3), (39936, 3), (39937, 3), (159744, 3), (159744, 4),
                                   (159745, 3)])
def test_sample_phase_sizes(n, per):
    print("sample phase", n, per, flush=True)
    X, eps, want = groups(n, per)
    args = (eps, 1.0, 1, 2, 1.0, 4, True)
    if n < 40000:
        # groups are the oracle's clusters: every pair in one is within eps,
        # every other is not
        ref = O.run_ref(X, *args)
        assert ref.subspaces == [[0], [1], [0, 1]]
        for a, b in zip(ref.labels, want):
            assert np.array_equal(O.canonical(a), O.canonical(b))
    got = INSCY.run(torch.from_numpy(X).cuda(), *args, 0, mode=_lib.MODE_BATCHED)
    assert got.subspaces == [[0], [1], [0, 1]]
    for a, b in zip(got.labels, want):
        assert np.array_equal(a, O.canonical(b))


# the permuted level orders' passes over one pair, a few and all pairs of a level at once
@pytest.mark.parametrize("order", [1, -1])
@pytest.mark.parametrize("max_batch", [1, 3, 0])
def test_permuted_order_in_batches_matches_oracle(max_batch, order):
    for n, d, eps, num_obj, rect in ((257, 5, 0.11, 4, True), (1201, 4, 0.05, 4, False), (1031, 7, 0.07, 2, True)):
        print("permuted batches", max_batch, order, n, d, flush=True)
        X = edge_data(n + d, n, d, eps)
        args = (eps, 1.0, num_obj, max(4, n // 40), 1.0, 3, rect)
        ref = O.run_ref(X, *args, order, trace=True)
        _lib.set_tuning(max_batch=max_batch)
        _lib.debug_trace(True)
        try:
            got = INSCY.run(torch.from_numpy(X).cuda(), *args, order, mode=_lib.MODE_BATCHED)
            trace = _lib.debug_trace_rows()
        finally:
            _lib.debug_trace(False)
            _lib.set_tuning()
        assert got.subspaces == ref.subspaces
        for a, b in zip(ref.labels, got.labels):
            assert np.array_equal(O.canonical(a), b)
        assert np.array_equal(trace, ref.trace)


def clumps(n, d, eps, dims, seed):
    """Uniform points with three groups that are dense in `dims` dimensions each."""
    rng = np.random.default_rng(seed)
    X = rng.random((n, d)).astype(np.float32)
    for c in range(3):
        rows = np.arange(c * n // 4, (c + 1) * n // 4)[:, None]
        at = np.sort(rng.choice(d, dims, replace=False)) if c else np.r_[0:dims - 1, d - 1]
        size = (c + 1) * n // 4 - c * n // 4
        X[rows, at] = (rng.uniform(0.2, 0.8, dims) + 0.4 * eps * rng.standard_normal((size, dims))).astype(np.float32)
    return np.clip(X, 0.0, 1.0)


def traced(X, args):
    _lib.debug_trace(True)
    try:
        got = INSCY.run(torch.from_numpy(X).cuda(), *args, mode=_lib.MODE_BATCHED)
        return got, _lib.debug_trace_rows()
    finally:
        _lib.debug_trace(False)


def by_child(X, args, generic):
    """The run with one walk per child, compiled for its k or not."""
    _lib.debug_walk_per_child(True)
    _lib.debug_generic_walk(generic)
    try:
        return traced(X, args)
    finally:
        _lib.debug_generic_walk(False)
        _lib.debug_walk_per_child(False)


# one walk per mask, one per child (compiled for its k, and for any k): the same
# trees and labels
@pytest.mark.parametrize("n,d,eps,dims", [(350, 9, 0.04, 5), (1203, 7, 0.01, 4)])
@pytest.mark.parametrize("rect", [True, False])
def test_walks_per_mask_and_per_child_agree(n, d, eps, dims, rect):
    print("walk routes", n, d, eps, rect, flush=True)
    X = clumps(n, d, eps, dims, n * d)
    args = (eps, 1.0, 4, n // 6, 1.0, 4, rect, 0)
    a, ta = traced(X, args)
    for generic in (False, True):
        b, tb = by_child(X, args, generic)
        # a walk per child leaves out the points that the counts of smaller
        # subspaces decide, a walk per mask does not look them up
        assert b.stats["queries"] < a.stats["queries"]
        assert a.subspaces == b.subspaces and np.array_equal(a.labels, b.labels)
        assert np.array_equal(ta, tb)


def many_groups(n, d, c, eps, seed):
    """Half of the points at the upper edge of each dimension's first cell (all of
    them on s-connection chains), the others in the middles of the other cells: every
    tree splits into c - 1 groups, and a chain passes to most."""
    rng = np.random.default_rng(seed)
    # the larger the first cell's share, the smaller the dimension's entropy
    cell = np.where(rng.random((n, d)) < np.linspace(0.4, 0.6, d), 0, rng.integers(1, c, (n, d)))
    off = np.where(cell == 0, 1 - (0.5 + 0.4 * rng.uniform(-1, 1, (n, d))) * eps * c,
                   0.5 + 0.1 * rng.uniform(-1, 1, (n, d)))
    return ((cell + off) / c).astype(np.float32)


# permuted level orders where a chain passes to most groups: a batch keeps to its
# bytes (and as many again for its children's prunes), whatever they come to
@pytest.mark.parametrize("order", [1, -1])
@pytest.mark.parametrize("n,d,c,budget", [(1500, 4, 20, 1 << 20), (1500, 4, 20, 1 << 19), (900, 5, 10, 1 << 19)])
def test_permuted_batches_keep_to_their_budget(n, d, c, budget, order):
    print("permuted budget", n, d, c, budget, order, flush=True)
    # levels against the dimensions: chains lie above the levels restricted first
    X = np.ascontiguousarray(many_groups(n, d, c, 0.01, n)[:, ::order])
    args = (0.01, 1.0, 4, 30, 1.0, c, True, order)
    ref = O.run_ref(X, *args[:7], order, trace=True)
    whole = None
    for b in (0, budget):
        _lib.debug_batch_budget(b)
        try:
            got, trace = traced(X, args)
            most = _lib.debug_batch_most()
        finally:
            _lib.debug_batch_budget(0)
        print("bytes of a batch", b, most, flush=True)
        assert got.subspaces == ref.subspaces
        for r, g in zip(ref.labels, got.labels):
            assert np.array_equal(O.canonical(r), g)
        assert np.array_equal(trace, ref.trace)
        if whole is None:
            whole = most
        else:
            assert most <= 2 * budget + (1 << 18) < whole


# a permuted order's root lists, where points times dimensions pass what their
# positions hold: sized by the chains there are, refused past the limit
def test_permuted_root_lists_at_the_limit():
    n, d, c = 900, 5, 10
    X = many_groups(n, d, c, 0.01, n)
    args = (0.01, 1.0, 4, 30, 1.0, c, True, 1)
    ref = O.run_ref(X, *args[:7], 1)
    # near-edge marks: within eps of a cell's upper edge, the last cell's apart
    cell = np.minimum((X.astype(np.float64) * c).astype(int), c - 1)
    chains = int(((cell < c - 1) & ((cell + 1) / c - X < 0.01)).sum())
    assert n * d // 4 < chains < n * d
    try:
        for limit, fits in ((n * d, True), (chains + 40, True), (chains - 40, False)):
            print("chain limit", limit, chains, flush=True)
            _lib.debug_chain_limit(limit)
            if fits:
                got = INSCY.run(torch.from_numpy(X).cuda(), *args, mode=_lib.MODE_BATCHED)
                assert got.subspaces == ref.subspaces
                for r, g in zip(ref.labels, got.labels):
                    assert np.array_equal(O.canonical(r), g)
            else:
                with pytest.raises(_lib.InscyError) as e:
                    INSCY.run(torch.from_numpy(X).cuda(), *args, mode=_lib.MODE_BATCHED)
                assert e.value.code == _lib.INSCY_ERR_UNSUPPORTED
    finally:
        _lib.debug_chain_limit(0)


# every route of one run gives one result: a walk per mask and per child, compiled
# and not; one child subspace at a time, a few and all of a level; no index kept
# from one batch for the next; small batches
@pytest.mark.parametrize("rect,order", [(True, 0), (False, 0), (True, 1), (False, -1)])
def test_routes_give_one_result(rect, order):
    print("routes", rect, order, flush=True)
    w = datagen.small(5, n=4000, d=8, n_clusters=4, eps=0.02, cells=5, num_obj=4, min_size=60, sub_dims=(3, 5))
    args = (w.eps, w.F, w.num_obj, w.min_size, w.r, w.cells, rect, order)
    a, ta = traced(w.X, args)
    assert max(len(s) for s in a.subspaces) >= 3
    for child, generic, max_batch, keep, budget in ((True, False, 0, -1, 0), (True, True, 0, -1, 0),
                                                    (False, True, 0, -1, 0), (False, False, 1, -1, 0),
                                                    (True, False, 1, -1, 0), (False, False, 3, 0, 0),
                                                    (True, True, 0, 0, 0), (False, False, 0, 1 << 20, 2 << 20)):
        print("route", child, generic, max_batch, keep, budget, flush=True)
        _lib.debug_walk_per_child(child)
        _lib.debug_generic_walk(generic)
        _lib.set_tuning(max_batch=max_batch)
        _lib.debug_keep_budget(keep)
        _lib.debug_batch_budget(budget)
        try:
            b, tb = traced(w.X, args)
        finally:
            _lib.debug_batch_budget(0)
            _lib.debug_keep_budget(-1)
            _lib.set_tuning()
            _lib.debug_generic_walk(False)
            _lib.debug_walk_per_child(False)
        assert a.subspaces == b.subspaces and np.array_equal(a.labels, b.labels)
        assert np.array_equal(ta, tb)
        assert a.stats["trees"] == b.stats["trees"] and a.stats["calls"] == b.stats["calls"]


# the same sizes in the phi density (the groups' points meet its thresholds too;
# the oracle says so for the small ones)
@pytest.mark.parametrize("n,per", [(75, 3), (1025, 3), (39936, 3), (39937, 3), (159744, 3), (159744, 4), (159745, 3)])
def test_sample_phase_sizes_phi(n, per):
    print("sample phase phi", n, per, flush=True)
    X, eps, want = groups(n, per)
    args = (eps, 1.0, 1, 2, 1.0, 4, False)
    if n < 5000:
        ref = O.run_ref(X, *args)
        assert ref.subspaces == [[0], [1], [0, 1]]
        for a, b in zip(ref.labels, want):
            assert np.array_equal(O.canonical(a), O.canonical(b))
    got = INSCY.run(torch.from_numpy(X).cuda(), *args, 0, mode=_lib.MODE_BATCHED)
    assert got.subspaces == [[0], [1], [0, 1]]
    for a, b in zip(got.labels, want):
        assert np.array_equal(a, O.canonical(b))


# walks of up to 32 children against the oracle, and of up to 64 and (in two
# walks) 79 against the walk per child
@pytest.mark.parametrize("n,d,eps,dims", [(90, 20, 0.03, 3), (301, 33, 0.02, 4), (250, 60, 0.02, 3),
                                          (240, 80, 0.02, 3)])
@pytest.mark.parametrize("rect", [True, False])
def test_walks_of_more_than_16_children(n, d, eps, dims, rect):
    print("many children", n, d, eps, dims, rect, flush=True)
    X = clumps(n, d, eps, dims, n * d)
    args = (eps, 1.0, 4, n // 6, 1.0, 4, rect, 0)
    got, trace = traced(X, args)
    assert max(len(s) for s in got.subspaces) >= dims - 1
    if d == 20:
        ref = O.run_ref(X, *args[:7], 0, trace=True)
        assert got.subspaces == ref.subspaces
        for a, b in zip(ref.labels, got.labels):
            assert np.array_equal(O.canonical(a), b)
        assert np.array_equal(trace, ref.trace)
    b, tb = by_child(X, args, False)
    assert got.subspaces == b.subspaces and np.array_equal(got.labels, b.labels)
    assert np.array_equal(trace, tb)


def test_threads_share_streams_while_memory_is_released():
    # callers without a stream take one from the pool and give it back, from
    # several threads at once, while another returns the pools' idle contents
    import threading
    jobs = []
    for seed, n in enumerate((150, 700, 1501)):
        w = datagen.small(seed + 20, n=n, d=5, n_clusters=3, eps=0.04, min_size=max(5, n // 40))
        args = (w.eps, w.F, w.num_obj, w.min_size, w.r, w.cells, True, 0)
        jobs.append((w.X, args, INSCY.run(w.X, *args)))
    bad, stop = [], threading.Event()

    def work(k):
        try:
            for i in range(12):
                X, args, want = jobs[(k + i) % len(jobs)]
                got = INSCY.run(X if i % 2 else torch.from_numpy(X).cuda(), *args)
                if got.subspaces != want.subspaces or not np.array_equal(got.labels, want.labels):
                    bad.append((k, i))
        except Exception as e:  # noqa: BLE001
            bad.append((k, repr(e)))

    def release():
        while not stop.is_set():
            _lib.lib().inscy_release_memory()
            stop.wait(0.002)

    print("threads", flush=True)
    th = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    rel = threading.Thread(target=release)
    rel.start()
    for t in th:
        t.start()
    for t in th:
        t.join()
    stop.set()
    rel.join()
    assert not bad, bad
