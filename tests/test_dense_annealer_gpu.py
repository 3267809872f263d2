"""GPU parity of the rocm dense annealer against the CPU oracle.

Bit-exact cases use integer-valued W (J quarter-integral, every field and
energy exact in float) and the device MT19937 stream (rng=mt19937), which
replays the serial CPU annealer's random stream; the oracle is the C
restatement of CPUDenseGraphAnnealer (oracle/).  Float cases compare energies
with an FP64 recompute within stated tolerances.
"""
import numpy as np
import pytest

from problems import dense_int_W, dense_normal_W, schedule, SEED_BASE, dense_graph_8x8

pytestmark = pytest.mark.gpu

BETA = 50.0


@pytest.fixture(scope="module")
def rocm():
    import sqaod_amd.rocm as rocm
    return rocm


def make_pair(oracle, rocm, W, m, seed, algo="coloring", dtype=np.float32, **prefs):
    N = W.shape[0]
    ora = oracle.DenseGraphAnnealer(dtype, 1)
    ora.seed(seed)
    ora.set_qubo(W.astype(dtype))
    ora.set_m(m)
    ora.set_algorithm({"coloring": 3, "sa_naive": 6}[algo])
    ora.prepare()
    ora.randomize_spin()
    an = rocm.dense_graph_annealer(W.astype(dtype), dtype=dtype, n_trotters=m, algorithm=algo,
                                   rng="mt19937", **prefs)
    an.seed(seed)
    an.prepare()
    an.randomize_spin()
    return ora, an


def q_of(an):
    return np.stack(an.get_q())


@pytest.mark.parametrize("variant", [dict(), dict(field_precision="bf16x2"), dict(field_precision="fp8"),
                                     dict(sweep="plain"), dict(slices_per_block=1),
                                     dict(sweep_launch="cooperative")])
def test_config1_bit_exact_trajectory(oracle, rocm, variant):
    """N=128, m=32, integer W in [-8, 8], G 5.0 -> 0.01 (x0.97), beta=50: the
    spins of every slice and the energies equal the serial CPU annealer's
    after every step of the schedule."""
    N, m = 128, 32
    W = dense_int_W(N, SEED_BASE)
    ora, an = make_pair(oracle, rocm, W, m, seed=1000, **variant)
    assert np.array_equal(q_of(an), ora.get_q()), "randomize_spin differs"
    for step, G in enumerate(schedule()):
        ora.anneal_one_step(G, BETA)
        an.anneal_one_step(G, BETA)
        if step % 10 == 0 or step == len(schedule()) - 1:
            qa, qo = q_of(an), ora.get_q()
            assert np.array_equal(qa, qo), f"step {step}: {np.sum(qa != qo)} spins differ"
    an.make_solution()
    E = an.get_E()
    assert np.array_equal(E, ora.calculate_E())
    x = np.stack(an.get_x())
    assert np.array_equal(x, (ora.get_q() + 1) // 2)


@pytest.mark.parametrize("N,m", [(100, 5), (64, 2), (37, 3), (200, 7), (256, 16), (1, 1), (1, 3), (2, 1),
                                 (33, 1)])
def test_odd_shapes_bit_exact(oracle, rocm, N, m):
    """odd m (ring neighbours 0 and m-1 share a colour), m = 2 (both
    neighbours one slice), m = 1 (the slice is its own neighbour), N = 1 and N
    not a multiple of 32: bit-exact over 30 steps."""
    W = dense_int_W(N, SEED_BASE + N + m)
    ora, an = make_pair(oracle, rocm, W, m, seed=7 + m)
    for G in schedule()[:30]:
        ora.anneal_one_step(G, BETA)
        an.anneal_one_step(G, BETA)
    assert np.array_equal(q_of(an), ora.get_q())


def test_sa_naive_bit_exact(oracle, rocm):
    """m = 1 selects SA (CPUDenseGraphAnnealer.cpp:174-175); kT = G."""
    N, m = 96, 1
    W = dense_int_W(N, SEED_BASE + 5)
    ora, an = make_pair(oracle, rocm, W, m, seed=3, algo="sa_naive")
    assert an.get_preferences()["algorithm"] == "sa_naive"
    for kT in np.geomspace(20.0, 0.05, 60):
        ora.anneal_one_step(kT, 0.0)
        an.anneal_one_step(kT, 0.0)
    assert np.array_equal(q_of(an), ora.get_q())


def test_maximize_bit_exact(oracle, rocm):
    N, m = 64, 8
    W = dense_int_W(N, SEED_BASE + 9)
    ora = oracle.DenseGraphAnnealer(np.float32, 1)
    ora.seed(11)
    ora.set_qubo(W, oracle.MAXIMIZE)
    ora.set_m(m)
    ora.prepare()
    ora.randomize_spin()
    import sqaod_amd as sq
    an = rocm.dense_graph_annealer(W, sq.maximize, dtype=np.float32, n_trotters=m, rng="mt19937")
    an.seed(11)
    an.prepare()
    an.randomize_spin()
    for G in schedule()[:40]:
        ora.anneal_one_step(G, BETA)
        an.anneal_one_step(G, BETA)
    assert np.array_equal(q_of(an), ora.get_q())
    assert np.array_equal(an.get_E(), ora.calculate_E())


def test_float_energy_fp64(oracle, rocm):
    """W ~ N(0,1): get_E is the FP64 recompute rounded to float; it agrees
    with the oracle's FP64 energy of the same spins within 1e-5 relative."""
    N, m = 512, 16
    W = dense_normal_W(N, SEED_BASE + 2)
    an = rocm.dense_graph_annealer(W, dtype=np.float32, n_trotters=m)
    an.seed(5)
    an.prepare()
    an.randomize_spin()
    for G in schedule()[:50]:
        an.anneal_one_step(G, BETA)
    E = an.get_E()
    q = np.stack(an.get_q())
    h, J, c = oracle.dense_hamiltonian(W.astype(np.float64))
    Eref = oracle.dense_energy_q(h, J, c, q)
    assert np.allclose(E, Eref, rtol=1e-5, atol=1e-3)


def test_local_vs_plain_float(rocm):
    """The local-field sweep and the plain per-attempt-dot sweep make the same
    decisions on float data with the same stream (fields agree to rounding)."""
    N, m = 256, 8
    W = dense_normal_W(N, SEED_BASE + 3)
    res = []
    for sweep in ("local", "plain"):
        an = rocm.dense_graph_annealer(W, dtype=np.float32, n_trotters=m, sweep=sweep)
        an.seed(21)
        an.prepare()
        an.randomize_spin()
        for G in schedule()[:20]:
            an.anneal_one_step(G, BETA)
        res.append(np.stack(an.get_q()))
    frac = np.mean(res[0] != res[1])
    assert frac < 0.05


def test_known_answers(rocm):
    """sqaodpy/tests/test_dense_graph_annealer.py:85-96 and :154-178."""
    N = 8
    an = rocm.dense_graph_annealer(np.ones((N, N), np.float32), dtype=np.float32, n_trotters=1)
    an.prepare()
    an.set_q(np.ones(N, np.int8))
    E = an.get_E()
    assert len(E) == 1 and E[0] == N * N
    x = an.get_x()
    assert len(x) == 1 and np.all(x[0] == 1)
    an.set_q(-np.ones(N, np.int8))
    assert an.get_E()[0] == 0.


def test_trivial_problem_reaches_zero(rocm):
    """test_dense_graph_annealer.py:180-260: W = ones(10); minimize reaches E=0."""
    import sqaod_amd as sq
    for opt, sign in ((sq.minimize, 1), (sq.maximize, -1)):
        W = sign * np.ones((10, 10), np.float64)
        an = rocm.dense_graph_annealer(W, opt, dtype=np.float64, n_trotters=4)
        an.seed(0)
        an.prepare()
        an.randomize_spin()
        G = 5.0
        while G > 0.02:
            an.anneal_one_step(G, 1. / 0.03)
            G *= 0.95
        an.make_solution()
        E = an.get_E()
        assert np.min(E) == 0 if opt is sq.minimize else np.max(E) == 0


def test_8x8_example(rocm, oracle):
    W = dense_graph_8x8(np.float32)
    Emin, _ = oracle.dense_bf_search(W.astype(np.float64))
    an = rocm.dense_graph_annealer(W, dtype=np.float32, n_trotters=4)
    an.seed(1)
    an.prepare()
    an.randomize_spin()
    for G in schedule():
        an.anneal_one_step(G, BETA)
    assert np.min(an.get_E()) == Emin


def test_large_instance_runs(rocm, oracle):
    """N=2048, m=64, W ~ N(0,1): the sweep completes (no neighbour-wait
    abort), the energy decreases, and E agrees with an FP64 recompute."""
    N, m = 2048, 64
    W = dense_normal_W(N, SEED_BASE + 4)
    an = rocm.dense_graph_annealer(W, dtype=np.float32, n_trotters=m)
    an.seed(3)
    an.prepare()
    an.randomize_spin()
    E0 = np.mean(an.get_E())
    for G in schedule()[:40]:
        an.anneal_one_step(G, BETA)
    E1 = an.get_E()
    assert np.mean(E1) < E0
    q = np.stack(an.get_q())
    h, J, c = oracle.dense_hamiltonian(W.astype(np.float64))
    Eref = oracle.dense_energy_q(h, J, c, q)
    assert np.allclose(E1, Eref, rtol=1e-5, atol=1e-2)
    cnt = an.get_counters()
    assert cnt["flips"] > 0 and cnt["batches"] > 0


@pytest.mark.parametrize("N,m,spb,algo", [(1, 3, 1, "coloring"), (37, 3, 2, "coloring"), (63, 5, 4, "coloring"),
                                          (257, 6, 2, "coloring"), (1025, 3, 1, "coloring"),
                                          (200, 5, 4, "sa_naive")])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_one_wave_sweep_bit_exact(oracle, rocm, N, m, spb, algo, dtype):
    """The single-flip kernel of one wave a slice, which runs where teams do not
    fit, at the shapes of the team sweep's own test."""
    W = dense_int_W(N, SEED_BASE + 7 * N + m)
    ora, an = make_pair(oracle, rocm, W, m, seed=11 + N, algo=algo, dtype=dtype, multi_flip="off",
                        helper_wave="off", slices_per_block=spb)
    for G in (np.geomspace(20.0, 0.05, 30) if algo == "sa_naive" else schedule()[:160:5]):
        beta = 0.0 if algo == "sa_naive" else BETA
        ora.anneal_one_step(G, beta)
        an.anneal_one_step(G, beta)
        assert np.array_equal(q_of(an), ora.get_q())
    assert np.array_equal(an.get_E(), ora.calculate_E())


@pytest.mark.parametrize("form", ["fp32", "bf16x2", "fp8"])
def test_largest_lds_resident_n_bit_exact(oracle, rocm, form):
    """N = 11520, the largest padded N whose float local-field sweep fits one
    workgroup's LDS (fields, staged row, pending table, spin bits, neighbour
    mirrors and windows: 12.4 bytes per site plus fixed parts, within 160 KiB),
    m = 4: spins equal the serial CPU annealer's after three steps.  The row
    DMA then spans 45 1-KiB ops (46 counted ops after the prefetch group) and
    the pending table is 4096 entries for 11520 sites."""
    N, m = 11520, 4
    W = dense_int_W(N, SEED_BASE + 11)
    ora, an = make_pair(oracle, rocm, W, m, seed=321, field_precision=form)
    for G in schedule()[:3]:
        ora.anneal_one_step(G, BETA)
        an.anneal_one_step(G, BETA)
        qa, qo = q_of(an), ora.get_q()
        assert np.array_equal(qa, qo), f"{np.sum(qa != qo)} spins differ"


def test_spin_limit_gives_up_cleanly(rocm):
    """With a spin limit of one blocked iteration (forced from the host) the
    sweep's bounded wait gives up instead of waiting: the step raises
    RuntimeError, every kernel has exited, and the annealer works again once
    its spins are set anew."""
    W = dense_int_W(128, SEED_BASE + 41)
    an = rocm.dense_graph_annealer(W, dtype=np.float32, n_trotters=2, spin_limit=1)
    an.seed(3)
    an.prepare()
    an.randomize_spin()
    with pytest.raises(RuntimeError, match="spin limit"):
        for G in schedule()[:40]:
            an.anneal_one_step(G, BETA)
        an.get_q()  # a flag written by the last step is reported here at the latest
    with pytest.raises(RuntimeError):
        an.set_preferences(spin_limit=0)
    an.set_preferences(spin_limit=1 << 20)
    an.randomize_spin()
    for G in schedule()[:10]:
        an.anneal_one_step(G, BETA)
    an.make_solution()
    x = np.stack(an.get_x()).astype(np.float64)
    assert np.array_equal(an.get_E(), np.einsum("yi,yi->y", x @ W.astype(np.float64), x).astype(np.float32))


@pytest.mark.parametrize("T,N,m", [(8, 128, 32), (3, 128, 32), (16, 100, 7), (4, 64, 5), (2, 50, 2)])
def test_openmp_worker_streams_bit_exact(oracle, rocm, T, N, m):
    """sqaod.cpu's default on a multi-core host is the OpenMP coloring step
    (CPUDenseGraphAnnealer.cpp:303-339) with one MT19937 per worker seeded
    s + 17 w (:29-33) and the slices of each colour in static chunks; with
    n_workers = T the device replays that trajectory (the oracle's
    restatement with T workers): spins after every 10th step of the
    schedule, and the energies, bit for bit.  Odd m puts slice m-1 on worker
    0 between the colours; T above m/2 leaves workers without slices."""
    W = dense_int_W(N, SEED_BASE + 90 + T + m)
    ora = oracle.DenseGraphAnnealer(np.float32, T)
    ora.seed(1000)
    ora.set_qubo(W)
    ora.set_m(m)
    ora.prepare()
    ora.randomize_spin()
    an = rocm.dense_graph_annealer(W, dtype=np.float32, n_trotters=m, rng="mt19937", n_workers=T)
    assert an.get_preferences()["n_workers"] == T
    an.seed(1000)
    an.prepare()
    an.randomize_spin()
    assert np.array_equal(q_of(an), ora.get_q())
    for k, G in enumerate(schedule()[:100]):
        ora.anneal_one_step(G, BETA)
        an.anneal_one_step(G, BETA)
        if k % 10 == 0:
            assert np.array_equal(q_of(an), ora.get_q()), f"step {k}"
    assert np.array_equal(q_of(an), ora.get_q())
    assert np.array_equal(an.get_E(), ora.calculate_E())


def test_generators_continue_across_prepare(oracle, rocm):
    """prepare() called again does not restart the random streams (the CPU
    annealer seeds only in seed(), CPUDenseGraphAnnealer.cpp:29-33, 164-167):
    the reference tests' calling sequence prepare / randomize_spin / anneal,
    twice (test_dense_graph_annealer.py:356-361), stays bit-exact."""
    N, m = 60, 6
    W = dense_int_W(N, SEED_BASE + 97)
    ora, an = make_pair(oracle, rocm, W, m, seed=4)
    for rep in range(2):
        if rep:
            ora.prepare()
            ora.randomize_spin()
            an.prepare()
            an.randomize_spin()
        for G in schedule()[:15]:
            ora.anneal_one_step(G, BETA)
            an.anneal_one_step(G, BETA)
        assert np.array_equal(q_of(an), ora.get_q()), rep


@pytest.mark.parametrize("N,m,form,algo", [(128, 32, "fp32", "coloring"), (128, 32, "bf16x2", "coloring"),
                                           (128, 32, "fp8", "coloring"),
                                           (300, 7, "fp32", "coloring"), (64, 2, "fp32", "coloring"),
                                           (1000, 16, "bf16x2", "coloring"), (96, 1, "fp32", "sa_naive"),
                                           (2048, 64, "fp32", "coloring"), (5000, 4, "fp32", "coloring"),
                                           (6000, 3, "bf16x2", "coloring")])
def test_multi_flip_batches_bit_exact(oracle, rocm, N, m, form, algo):
    """multi_flip: a batch resolves all its accepted flips in order (each
    flip corrects the later lanes' fields with the gathered submatrix and the
    rows are applied in flip order), so the trajectory is still the serial
    CPU annealer's, bit for bit, in the flip-heavy start of the schedule and
    to its end.  N = 5000 and 6000 leave LDS for three and two row stage
    buffers (four at N <= 4096), so batches with more flips than buffers
    apply their earlier rows at once and defer fewer."""
    W = dense_int_W(N, SEED_BASE + 3 * N + m)
    # threshold 2: every batch after one with two accepting lanes is a multi-flip batch
    ora, an = make_pair(oracle, rocm, W, m, seed=31 + m, algo=algo, field_precision=form, multi_flip="2")
    assert an.get_preferences()["multi_flip"] == "2"
    sch = schedule() if N <= 300 else schedule()[:40]
    if algo == "sa_naive":
        sch = list(np.geomspace(20.0, 0.05, 60))
    for k, G in enumerate(sch):
        beta = 0.0 if algo == "sa_naive" else BETA
        ora.anneal_one_step(G, beta)
        an.anneal_one_step(G, beta)
        if k % 10 == 0 or k == len(sch) - 1:
            qa, qo = q_of(an), ora.get_q()
            assert np.array_equal(qa, qo), f"step {k}: {int(np.sum(qa != qo))} spins differ"
    assert np.array_equal(an.get_E(), ora.calculate_E())
    c = an.get_counters()
    assert c["flips"] > 0


@pytest.mark.parametrize("N,m", [(5000, 4), (6000, 3), (2048, 16)])
def test_multi_flip_engages_and_matches_single_flip(rocm, N, m):
    """The multi-flip sweep takes over where LDS holds at least two row stage
    buffers (four at N = 2048, three at 5000, two at 6000): in the flip-heavy
    first steps it commits the same spins as the single-flip sweep in fewer
    batches."""
    W = dense_int_W(N, SEED_BASE + 7 * N)
    runs = {}
    for mode in ("off", "2"):
        an = rocm.dense_graph_annealer(W, dtype=np.float32, n_trotters=m, multi_flip=mode)
        an.seed(5)
        an.prepare()
        an.randomize_spin()
        for G in schedule()[:3]:
            an.anneal_one_step(G, BETA)
        runs[mode] = (q_of(an), an.get_counters())
    assert np.array_equal(runs["off"][0], runs["2"][0])
    assert runs["2"][1]["flips"] == runs["off"][1]["flips"]
    assert runs["2"][1]["batches"] < 0.8 * runs["off"][1]["batches"]


@pytest.mark.parametrize("N,m,form,algo", [(128, 32, "fp32", "coloring"), (300, 7, "fp32", "coloring"),
                                           (1000, 16, "bf16x2", "coloring"), (96, 1, "fp32", "sa_naive"),
                                           (4096, 8, "fp32", "coloring"), (6000, 3, "bf16x2", "coloring")])
def test_helper_wave_bit_exact(oracle, rocm, N, m, form, algo):
    """helper_wave=on (the default): a team of four waves per slice sweeps it,
    one deciding, one adding the last flip's J row to the LDS fields, one
    preparing the attempts ahead, one reading the neighbours' decisions.  With
    multi_flip=off every sweep runs that kernel, and the trajectory is still
    the serial CPU annealer's, bit for bit."""
    W = dense_int_W(N, SEED_BASE + 5 * N + m)
    ora, an = make_pair(oracle, rocm, W, m, seed=41 + m, algo=algo, field_precision=form, multi_flip="off",
                        helper_wave="on")
    assert an.get_preferences()["helper_wave"] == "on"
    sch = schedule() if N <= 300 else schedule()[:30]
    if algo == "sa_naive":
        sch = list(np.geomspace(20.0, 0.05, 60))
    for k, G in enumerate(sch):
        beta = 0.0 if algo == "sa_naive" else BETA
        ora.anneal_one_step(G, beta)
        an.anneal_one_step(G, beta)
        if k % 10 == 0 or k == len(sch) - 1:
            qa, qo = q_of(an), ora.get_q()
            assert np.array_equal(qa, qo), f"step {k}: {int(np.sum(qa != qo))} spins differ"
    assert np.array_equal(an.get_E(), ora.calculate_E())


def test_helper_wave_on_off_same_sweep(rocm):
    """The team changes who does what, not the sweep: one wave a slice commits
    the same spins, flips and energies (float normal W, so
    the fields carry rounding that any change of operation order would
    show).  Batch counts are not compared: where a batch ends depends on how
    far the neighbour slices have got, which is timing."""
    W = dense_normal_W(2048, SEED_BASE + 99)
    runs = {}
    for mode in ("off", "on"):
        an = rocm.dense_graph_annealer(W, dtype=np.float32, n_trotters=32, helper_wave=mode)
        an.seed(9)
        an.prepare()
        an.randomize_spin()
        for G in schedule()[:12]:
            an.anneal_one_step(G, BETA)
        runs[mode] = (q_of(an), an.get_counters(), an.get_E())
    assert np.array_equal(runs["off"][0], runs["on"][0])
    assert runs["off"][1]["flips"] == runs["on"][1]["flips"]
    assert np.array_equal(runs["off"][2], runs["on"][2])


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("helper", ["on", "off"])
@pytest.mark.parametrize("spb", [1, 2, 4])
def test_helper_wave_with_several_slices_per_block(oracle, rocm, spb, helper, dtype):
    """Several slices of a workgroup, each by a team or, with helper_wave=off, by
    one wave (in single-flip batches), with a last workgroup that
    is not full: the serial CPU annealer's trajectory."""
    N, m = 300, 7
    W = dense_int_W(N, SEED_BASE + 17 * spb)
    ora, an = make_pair(oracle, rocm, W, m, seed=61 + spb, dtype=dtype, slices_per_block=spb, helper_wave=helper,
                        **({} if helper == "on" else {"multi_flip": "off"}))
    assert int(an.get_preferences()["slices_per_block"]) == spb
    for k, G in enumerate(schedule()[:30]):
        ora.anneal_one_step(G, BETA)
        an.anneal_one_step(G, BETA)
    assert np.array_equal(q_of(an), ora.get_q())
    assert np.array_equal(an.get_E(), ora.calculate_E())


def test_helper_wave_near_the_lds_limit(oracle, rocm):
    """N = 8192: fields, two row stage buffers, h and the tables by site (fewer
    slots than sites) fill most of a workgroup's 160 KiB of LDS, and the team
    sweep still runs the serial CPU annealer's trajectory."""
    N, m = 8192, 2
    W = dense_int_W(N, SEED_BASE + 8192)
    ora, an = make_pair(oracle, rocm, W, m, seed=73, multi_flip="off", helper_wave="on")
    for G in schedule()[:8]:
        ora.anneal_one_step(G, BETA)
        an.anneal_one_step(G, BETA)
    assert np.array_equal(q_of(an), ora.get_q())
    assert np.array_equal(an.get_E(), ora.calculate_E())


@pytest.mark.parametrize("N,m,spb,dtype,algo", [
    (5, 2, 2, np.float32, "coloring"), (63, 5, 4, np.float64, "coloring"), (65, 3, 1, np.float32, "coloring"),
    (255, 9, 3, np.float32, "coloring"), (257, 6, 2, np.float64, "coloring"), (1024, 4, 4, np.float32, "coloring"),
    (1025, 4, 2, np.float32, "coloring"), (1025, 3, 1, np.float64, "coloring"), (200, 5, 4, np.float64, "sa_naive")])
def test_team_sweep_bit_exact(oracle, rocm, N, m, spb, dtype, algo):
    """The team sweep at the sizes where its rings (256 prepared attempts),
    words of 16 decisions, chunks of 64 and tables by site (shared slots
    resolved up to N = 1024) wrap or change, 1 to 4 slices per workgroup with
    the ring of slices closing inside one or not, float and double: the serial
    CPU annealer's spins and energies, bit for bit."""
    W = dense_int_W(N, SEED_BASE + 7 * N + m)
    ora, an = make_pair(oracle, rocm, W, m, seed=11 + N, algo=algo, dtype=dtype, multi_flip="off",
                        slices_per_block=spb)
    for G in (np.geomspace(20.0, 0.05, 30) if algo == "sa_naive" else schedule()[:160:5]):
        beta = 0.0 if algo == "sa_naive" else BETA
        ora.anneal_one_step(G, beta)
        an.anneal_one_step(G, beta)
        assert np.array_equal(q_of(an), ora.get_q())
    assert np.array_equal(an.get_E(), ora.calculate_E())


@pytest.mark.parametrize("prefs", [dict(), dict(helper_wave="off"), dict(helper_wave="off", multi_flip="2"),
                                   dict(sweep="plain")], ids=["team", "one_wave", "multi_flip", "plain"])
@pytest.mark.parametrize("N,m", [(5, 64), (16, 48), (32, 33), (61, 48)])
def test_short_slices_over_many_blocks_bit_exact(oracle, rocm, N, m, prefs):
    """A slice this short may end before a neighbour in another block has
    started, which then reads its spins: those from before the sweep, to which
    it adds the published flips."""
    W = dense_int_W(N, SEED_BASE + 19 * N)
    ora, an = make_pair(oracle, rocm, W, m, seed=23 + N, slices_per_block=1, **prefs)
    for k, G in enumerate(schedule()):
        ora.anneal_one_step(G, BETA)
        an.anneal_one_step(G, BETA)
        if k % 20 == 0:
            assert np.array_equal(q_of(an), ora.get_q()), f"step {k}"
    assert np.array_equal(q_of(an), ora.get_q())


def test_spins_follow_through_changing_steps(oracle, rocm):
    """A sweep leaves its spins in another buffer than it read, the naive step,
    set_q and randomize_spin work on the present one: a mixed sequence of odd
    lengths stays the serial CPU annealer's."""
    N, m = 70, 6
    W = dense_int_W(N, SEED_BASE + 29)
    ora, an = make_pair(oracle, rocm, W, m, seed=37)
    rng = np.random.default_rng(SEED_BASE)
    for rep, steps in enumerate([1, 2, 3, 1, 4, 5]):
        for name, code in (("coloring", 3), ("naive", 2)):
            ora.set_algorithm(code)
            an.set_preferences(algorithm=name)
            for G in schedule()[rep * 20:rep * 20 + steps]:
                ora.anneal_one_step(G, BETA)
                an.anneal_one_step(G, BETA)
            assert np.array_equal(q_of(an), ora.get_q()), (rep, name)
            assert np.array_equal(an.get_E(), ora.calculate_E())
        if rep == 2:
            q = 2 * rng.integers(0, 2, N).astype(np.int8) - 1
            ora.set_q(np.tile(q, (m, 1)))
            an.set_q(q)
        elif rep == 4:
            ora.randomize_spin()
            an.randomize_spin()
        assert np.array_equal(q_of(an), ora.get_q()), rep


@pytest.mark.parametrize("N,m,spb,dtype", [(4096, 300, 1, np.float32), (1024, 600, 2, np.float32),
                                           (2000, 500, 1, np.float64), (300, 1500, 1, np.float32)])
def test_more_slices_than_teams_fit(rocm, N, m, spb, dtype):
    """slices_per_block with more blocks than the team sweep has room for on the
    chip, which fit with one wave a slice (the last shape: several teams to a
    CU, more than there are CUs): the same spins as one wave a slice."""
    W = dense_int_W(N, SEED_BASE + 31).astype(dtype)
    runs = []
    for helper in ("on", "off"):
        an = rocm.dense_graph_annealer(W, dtype=dtype, n_trotters=m, slices_per_block=spb, helper_wave=helper,
                                       multi_flip="off")
        an.seed(41)
        an.prepare()
        an.randomize_spin()
        for G in (2.0, 0.5):
            an.anneal_one_step(G, BETA)
        runs.append(q_of(an))
    assert np.array_equal(runs[0], runs[1])


def test_refused_launch_is_reported_once(rocm):
    """More slices, one a block, than any sweep has room for: the step's launch
    is refused with an error, and the next solver's calls do not meet it again."""
    N, m = 4096, 1100
    an = rocm.dense_graph_annealer(dense_int_W(N, SEED_BASE + 53), dtype=np.float32, n_trotters=m, slices_per_block=1,
                                   multi_flip="off")
    an.seed(1)
    an.prepare()
    an.randomize_spin()
    with pytest.raises(RuntimeError, match="too many blocks"):
        an.anneal_one_step(1.0, BETA)
    rocm.dense_graph_bf_searcher(dense_graph_8x8(np.float32), dtype=np.float32).search()
    other = rocm.dense_graph_annealer(dense_int_W(64, SEED_BASE), dtype=np.float32, n_trotters=4)
    other.seed(1)
    other.prepare()
    other.randomize_spin()
    other.anneal_one_step(1.0, BETA)
    other.get_E()


@pytest.mark.parametrize("N,m,spb,mode", [(4096, 300, 1, "auto"), (1024, 2000, 0, "auto"), (2048, 600, 2, "on")])
def test_more_slices_than_multi_flip_blocks_fit(rocm, N, m, spb, mode):
    """The multi-flip sweep's stage buffers give way, to two and then to the
    single-flip sweep, where with them the blocks would not fit on the chip:
    the same spins as single-flip sweeps."""
    W = dense_int_W(N, SEED_BASE + 43)
    runs = []
    for multi in (mode, "off"):
        an = rocm.dense_graph_annealer(W, dtype=np.float32, n_trotters=m, slices_per_block=spb, helper_wave="off",
                                       multi_flip=multi)
        an.seed(47)
        an.prepare()
        an.randomize_spin()
        for G in (2.0, 0.5):
            an.anneal_one_step(G, BETA)
        runs.append(q_of(an))
    assert np.array_equal(runs[0], runs[1])


@pytest.mark.parametrize("N,spb,dtype", [(20, 0, np.float32), (100, 0, np.float32), (100, 0, np.float64),
                                         (100, 2, np.float32), (300, 1, np.float32), (1100, 0, np.float32)])
def test_one_slice_coloring_bit_exact(oracle, rocm, N, spb, dtype):
    """prepare() selects SA for one slice; the coloring algorithm asked for
    after it runs with the slice as its own neighbour on both sides, by the
    one-wave kernel."""
    W = dense_int_W(N, SEED_BASE + 13 * N)
    ora, an = make_pair(oracle, rocm, W, 1, seed=17 + N, dtype=dtype, slices_per_block=spb)
    ora.set_algorithm(3)
    an.set_preferences(algorithm="coloring")
    assert an.get_preferences()["algorithm"] == "coloring"
    for G in schedule()[:160:5]:
        ora.anneal_one_step(G, BETA)
        an.anneal_one_step(G, BETA)
        assert np.array_equal(q_of(an), ora.get_q())


def test_team_sweep_after_a_tag_period_of_others(oracle, rocm):
    """A team sweep a whole tag period (2047 sweeps) after the last one, the
    sweeps in between by the one-wave kernel: no word of the old sweep counts."""
    N, m = 24, 4
    W = dense_int_W(N, SEED_BASE + 4)
    ora, an = make_pair(oracle, rocm, W, m, seed=6, multi_flip="off")
    for k in range(2060):
        an.set_preferences(helper_wave="off" if 2 <= k < 2048 else "on")
        G = 3.0 if k % 50 else 0.5
        ora.anneal_one_step(G, 1.0)
        an.anneal_one_step(G, 1.0)
        if k >= 2040:
            assert np.array_equal(q_of(an), ora.get_q()), k


def test_team_words_follow_the_number_of_slices(rocm):
    """The published words are kept through prepare() and made anew where the
    slices' number or length changes (the first change leaves their total as
    it was): the same spins as one wave a slice."""
    runs = []
    for helper in ("on", "off"):
        an = rocm.dense_graph_annealer(dense_int_W(100, SEED_BASE + 59), dtype=np.float32, helper_wave=helper)
        out = []
        for N, m in [(100, 8), (100, 8), (1500, 4), (100, 5), (600, 8), (100, 8)]:
            an.set_qubo(dense_int_W(N, SEED_BASE + 59))
            an.set_preferences(n_trotters=m)
            an.seed(3)
            an.prepare()
            an.randomize_spin()
            for G in (3.0, 0.5, 0.1):
                an.anneal_one_step(G, BETA)
            out.append(q_of(an))
        runs.append(out)
    assert all(np.array_equal(a, b) for a, b in zip(*runs))


def test_team_sweep_past_its_tag_period(oracle, rocm):
    """More sweeps than the published words have tags (2047)."""
    N, m = 24, 4
    W = dense_int_W(N, SEED_BASE + 3)
    ora, an = make_pair(oracle, rocm, W, m, seed=5, multi_flip="off")
    for k in range(2150):
        G = 3.0 if k % 50 else 0.5
        ora.anneal_one_step(G, 1.0)
        an.anneal_one_step(G, 1.0)
        if k > 2030 and k % 20 == 0:
            assert np.array_equal(q_of(an), ora.get_q()), k
    assert np.array_equal(q_of(an), ora.get_q())
