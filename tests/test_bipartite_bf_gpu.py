"""Bipartite brute-force searcher on the rocm device against the oracle's
restatement of the one-worker CPU search (CPUBipartiteGraphBFSearcher,
CPUBipartiteGraphBatchSearch) and the reference tests' known answers
(sqaodpy/tests/test_bipartite_graph_bf_searcher.py).  Integer data make every
energy exact, so minima and pair lists must be equal."""
import numpy as np
import pytest

from problems import SEED_BASE

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rocm():
    import sqaod_amd.rocm as rocm
    return rocm


def packed(x):
    x = np.asarray(x, np.uint64)
    N = x.shape[-1]
    return (x << np.arange(N - 1, -1, -1, dtype=np.uint64)).sum(axis=-1)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_known_answers(rocm, dtype):
    """test_bipartite_graph_bf_searcher.py:41-110."""
    s = rocm.bipartite_graph_bf_searcher(np.ones(4), np.ones(4), np.ones((4, 4)), optimize=1, dtype=dtype)
    s.search()
    E = s.get_E()
    assert len(E) == 1 and E[0] == 4 * 4 + 4 + 4
    x = s.get_x()
    assert len(x) == 1 and np.all(x[0][0] == 1) and np.all(x[0][1] == 1)
    assert s.get_problem_size() == (4, 4)
    for opt, sign, Eexp, bit in [(0, 1, 0, 0), (0, -1, -80, 1), (1, 1, 80, 1), (1, -1, 0, 0)]:
        s.set_qubo(sign * np.ones(8), sign * np.ones(8), sign * np.ones((8, 8)), opt)
        s.search()
        E, x = s.get_E(), s.get_x()
        assert E[0] == Eexp and len(x) == 1
        assert np.all(x[0][0] == bit) and np.all(x[0][1] == bit)


@pytest.mark.parametrize("N0,N1,T0,opt,seed", [(5, 4, 1024, 0, 1), (3, 7, 256, 1, 2), (10, 6, 256, 0, 3),
                                               (12, 8, 512, 1, 4), (14, 9, 1024, 0, 5), (10, 13, 256, 0, 6)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_matches_oracle(oracle, rocm, N0, N1, T0, opt, seed, dtype):
    """b0, b1, W integers in [-2, 2] (ties are common): Emin and the pair list
    equal the oracle's -- the first N0 + N1 minimisers in the order (x0 tile,
    x1, x0 in tile) -- including x0 tiles smaller than 2^N0 and searches
    that take several scan rectangles (N1 = 13: two x1 chunks)."""
    rng = np.random.default_rng(SEED_BASE + seed)
    b0 = rng.integers(-2, 3, N0).astype(np.float64)
    b1 = rng.integers(-2, 3, N1).astype(np.float64)
    W = rng.integers(-2, 3, (N1, N0)).astype(np.float64)
    Eo, xs0, xs1 = oracle.bipartite_bf_search(b0, b1, W, dtype=dtype, optimize=opt, tile_size0=T0)
    s = rocm.bipartite_graph_bf_searcher(b0, b1, W, optimize=opt, dtype=dtype, tile_size_0=T0)
    s.prepare()
    calls = 0
    while True:
        done, cx0, cx1 = s.search_range()
        calls += 1
        if done:
            break
    assert cx0 == 1 << N0 and cx1 == 0
    if N1 == 13:
        assert calls >= 2
    s.make_solution()
    E = s.get_E()
    x = s.get_x()
    assert E.dtype == dtype and np.all(E == Eo) and len(x) == len(xs0)
    assert np.array_equal(packed([p[0] for p in x]), xs0)
    assert np.array_equal(packed([p[1] for p in x]), xs1)


def test_all_ties_keep_first_pairs_in_visiting_order(oracle, rocm):
    N0, N1 = 9, 5
    z0, z1, zW = np.zeros(N0), np.zeros(N1), np.zeros((N1, N0))
    for T0 in (256, 512):
        Eo, xs0, xs1 = oracle.bipartite_bf_search(z0, z1, zW, tile_size0=T0)
        s = rocm.bipartite_graph_bf_searcher(z0, z1, zW, dtype=np.float32, tile_size_0=T0)
        s.search()
        x = s.get_x()
        assert len(x) == N0 + N1
        assert np.array_equal(packed([p[0] for p in x]), xs0)
        assert np.array_equal(packed([p[1] for p in x]), xs1)


def test_errors(rocm):
    s = rocm.bipartite_graph_bf_searcher(dtype=np.float32)
    with pytest.raises(RuntimeError):
        s.set_qubo(np.ones(64), np.ones(2), np.ones((2, 64)))
    with pytest.raises(RuntimeError):
        s.set_qubo(np.ones(3), np.ones(2), np.ones((3, 2)))
    with pytest.raises(RuntimeError):
        s.prepare()


def test_many_searchers_on_several_threads(rocm):
    """The minima and first pairs of a rectangle come back through staging memory
    of the device: more searchers than it keeps blocks for, on several threads
    at once, each find what they find alone."""
    from concurrent.futures import ThreadPoolExecutor
    rng = np.random.default_rng(SEED_BASE + 77)
    problems = [tuple(rng.integers(-3, 4, s).astype(np.float32) for s in (n0, n1, (n1, n0)))
                for n0, n1 in [(3 + k % 10, 2 + (3 * k) % 13) for k in range(24)]]

    def search(p):
        s = rocm.bipartite_graph_bf_searcher(*p, dtype=np.float32)
        for _ in range(3):
            s.search()
        return s, s.get_E(), s.get_x()

    alone = [search(p) for p in problems]
    with ThreadPoolExecutor(12) as pool:
        together = list(pool.map(search, problems))
    for (_, E0, x0), (_, E1, x1) in zip(alone, together):
        assert np.array_equal(E0, E1) and len(x0) == len(x1)
        assert all(np.array_equal(a, b) for p, q in zip(x0, x1) for a, b in zip(p, q))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("N0,N1", [(1, 1), (63, 1), (11, 5), (4, 12), (20, 1), (18, 13)])
def test_real_weights_take_the_least_over_x0(rocm, dtype, N0, N1):
    """N(0, 1) weights, where the minimum is one pair: the x0 of the negative
    sums of its x1, over one to many rectangles of high patterns (N0 = 63: the
    first rectangle alone, its high bits fixed at zero)."""
    rng = np.random.default_rng(SEED_BASE + 100 * N0 + N1)
    b0, b1, W = (rng.standard_normal(s).astype(dtype) for s in (N0, N1, (N1, N0)))
    s = rocm.bipartite_graph_bf_searcher(b0, b1, W, dtype=dtype)
    s.prepare()
    done, cx0, _ = s.search_range()
    while not done and N0 <= 20:
        done, cx0, _ = s.search_range()
    s.make_solution()
    x1 = ((np.arange(1 << N1)[:, None] >> np.arange(N1 - 1, -1, -1)) & 1).astype(np.float64)
    d = b0.astype(np.float64) + x1 @ W.astype(np.float64)
    if N0 == 63:
        d[:, packed(np.eye(N0, dtype=np.uint64)) >= cx0] = 0.0  # not reached
    E = np.minimum(d, 0.0).sum(axis=1) + x1 @ b1.astype(np.float64)
    best = int(np.argmin(E))
    x = s.get_x()
    assert len(x) == 1 and packed(x[0][1]) == best and np.array_equal(np.asarray(x[0][0]), (d[best] < 0).astype(np.int8))
    # (N0 + 1)(N1 + 1) terms summed in 64 bits in two orders, then one rounding to dtype
    sums = 2 * (N0 + 1) * (N1 + 1) * 2.0 ** -53 * sum(np.abs(v.astype(np.float64)).sum() for v in (b0, b1, W))
    assert abs(float(s.get_E()[0]) - E[best]) <= sums + np.finfo(dtype).eps / 2 * (abs(E[best]) + sums)
