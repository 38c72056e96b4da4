"""Walks on the GPU against the oracle: bit-exact paths for the same Philox stream and tables."""
import numpy as np
import pytest

from helpers import chi_square_p, graph_from_degrees, weights

pytestmark = pytest.mark.gpu


def run_offline(orc, xadj, adjncy, w, seeds, length, stop, seed):
    from skywalker_amd import capi
    g = capi.Graph.upload(xadj, adjncy, w)
    g.build_tables()
    prob, alias, valid = g.tables()
    paths_d, len_d, sampled, sec = g.walk_offline(seeds, length, stop, seed)
    paths, lengths = paths_d.to_host((len(seeds), length + 1)), len_d.to_host()
    g.free()
    opaths, olengths, osampled = orc.walk_offline(xadj, adjncy, prob, alias, seeds, length, stop, seed)
    return (paths, lengths, sampled), (opaths, olengths, osampled), (prob, alias, valid)


def test_config1_deepwalk_bit_exact(orc):
    xadj, adjncy = orc.rmat_csr(16, 16, 42)
    w = orc.gen_weights(orc.W_UNIFORM, 42, len(adjncy), 1.0, 100.0)
    seeds = orc.gen_seeds(42, 1 << 16, 4096)
    got, want, _ = run_offline(orc, xadj, adjncy, w, seeds, 80, 0.0, 42)
    assert np.array_equal(got[1], want[1])
    assert np.array_equal(got[0], want[0])
    assert got[2] == want[2] == int(want[1].sum())


def test_ppr_bit_exact_and_length_law(orc):
    # every vertex has out-edges so only the stop test ends a walk
    rng = np.random.default_rng(4)
    V = 2000
    xadj, adjncy, w = graph_from_degrees(rng.integers(1, 40, V), rng, "lognormal", V=V)
    seeds = rng.integers(0, V, 60000, dtype=np.uint32)
    tp, L = 0.15, 100
    got, want, _ = run_offline(orc, xadj, adjncy, w, seeds, L, tp, 7)
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1]) and got[2] == want[2]
    lengths = got[1].astype(np.float64)
    mean = (1 - (1 - tp) ** L) / tp - 1 + (1 - tp) ** L  # E[min(G, L)] with G ~ Geometric(tp) counting failures
    assert abs(lengths.mean() - mean) < 4 * np.sqrt((1 - tp) / tp**2 / len(seeds))
    k = np.arange(0, 30)
    cnt = np.array([(lengths == x).sum() for x in k])
    pk = tp * (1 - tp) ** k
    assert chi_square_p(np.append(cnt, len(seeds) - cnt.sum()), np.append(pk, 1 - pk.sum())) > 0.01


@pytest.mark.parametrize("n,length,stop", [(1, 1, 0.0), (63, 64, 0.0), (2048, 65, 0.02), (2049, 130, 0.0), (8192, 63, 0.15),
                                           (8193, 129, 0.02), (70, 200, 0.0)])
@pytest.mark.parametrize("index", [False, True])
def test_walkers_with_a_wavefront_each(orc, n, length, stop, index):
    # the limits between one walker to a wavefront and one to a lane, windows of 64 steps that end inside a walk, and
    # walks that end at rows without weight, without entries and at start vertices that do not exist
    from skywalker_amd import capi
    rng = np.random.default_rng(n)
    V = 3000
    xadj, adjncy, w = graph_from_degrees(np.append(rng.integers(0, 40, V - 1), 5000), rng, "sparse", V=V)
    w[xadj[10]:xadj[40]] = 0.0
    seeds = rng.integers(0, V + 20, n, dtype=np.uint32)
    g = capi.Graph.upload(xadj, adjncy, w)
    g.build_tables()
    if index:
        g.build_walk_index()
    prob, alias, _ = g.tables()
    paths_d, len_d, sampled, _ = g.walk_offline(seeds, length, stop, 11)
    paths, lengths = paths_d.to_host((n, length + 1)), len_d.to_host()
    g.free()
    opaths, olengths, osampled = orc.walk_offline(xadj, adjncy, prob, alias, seeds, length, stop, 11)
    assert np.array_equal(lengths, olengths) and sampled == osampled
    assert np.array_equal(paths, opaths)


@pytest.mark.parametrize("entries", [(4 << 20) // 8, (4 << 20) // 8 + 1])
@pytest.mark.parametrize("n,length", [(4096, 24), (4097, 23), (4097, 24), (8192, 70), (8193, 24)])
def test_thousands_of_walkers_with_a_wavefront_each(orc, n, length, entries):
    # where the tables take more than 4 MB and the walk has 24 steps or more, up to 8,192 walkers have a wavefront each: both sides
    # of each of the three limits
    from skywalker_amd import capi
    rng = np.random.default_rng(n + length)
    V = 20000
    degs = rng.integers(0, 50, V)
    degs[-1] = entries - degs[:-1].sum()
    xadj, adjncy, w = graph_from_degrees(degs, rng, "sparse", V=V)
    assert len(w) == entries and degs[-1] > 0
    w[xadj[10]:xadj[40]] = 0.0
    seeds = rng.integers(0, V + 20, n, dtype=np.uint32)
    g = capi.Graph.upload(xadj, adjncy, w)
    g.build_tables()
    prob, alias, _ = g.tables()
    paths_d, len_d, sampled, _ = g.walk_offline(seeds, length, 0.01, 13)
    paths, lengths = paths_d.to_host((n, length + 1)), len_d.to_host()
    g.free()
    opaths, olengths, osampled = orc.walk_offline(xadj, adjncy, prob, alias, seeds, length, 0.01, 13)
    assert np.array_equal(lengths, olengths) and sampled == osampled
    assert np.array_equal(paths, opaths)


def test_dead_ends_and_zero_weight_rows(orc):
    # path graph 0 -> 1 -> 2 -> 3 (3 has no out-edge); vertex 4 has one zero-weight edge; 5 loops on itself
    xadj = np.array([0, 1, 2, 3, 3, 4, 5], np.uint32)
    adjncy = np.array([1, 2, 3, 0, 5], np.uint32)
    w = np.array([1, 1, 1, 0, 2], np.float32)
    seeds = np.array([0, 1, 2, 3, 4, 5], np.uint32)
    got, want, _ = run_offline(orc, xadj, adjncy, w, seeds, 6, 0.0, 1)
    assert got[1].tolist() == [3, 2, 1, 0, 0, 6]
    assert got[0][0, :4].tolist() == [0, 1, 2, 3] and np.all(got[0][0, 4:] == 0xFFFFFFFF)
    assert np.all(got[0][5] == 5)
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])


def test_next_hop_frequencies_chi_square(orc):
    # star: hub 0 with 50 weighted spokes; one step from the hub must follow w / sum(w)
    rng = np.random.default_rng(8)
    d = 50
    xadj = np.zeros(d + 2, np.uint32)
    xadj[1:] = d
    adjncy = np.arange(1, d + 1, dtype=np.uint32)
    w = rng.lognormal(0, 1, d).astype(np.float32)
    N = 200000
    seeds = np.zeros(N, np.uint32)
    got, want, _ = run_offline(orc, xadj, adjncy, w, seeds, 1, 0.0, 3)
    assert np.array_equal(got[0], want[0])
    counts = np.bincount(got[0][:, 1], minlength=d + 1)[1:]
    assert chi_square_p(counts, w.astype(np.float64) / w.astype(np.float64).sum()) > 0.01


def test_walk_does_not_depend_on_batch_composition(orc):
    # walker i's path is a function of (seed, i, start vertex) only
    from skywalker_amd import capi
    xadj, adjncy = orc.rmat_csr(12, 8, 5)
    w = orc.gen_weights(orc.W_UNIT, 5, len(adjncy))
    g = capi.Graph.upload(xadj, adjncy, w)
    g.build_tables()
    seeds = orc.gen_seeds(1, 1 << 12, 3000)
    full = g.walk_offline(seeds, 20, 0.0, 9)[0].to_host((3000, 21))
    part = g.walk_offline(seeds[:1000], 20, 0.0, 9)[0].to_host((1000, 21))
    g.free()
    assert np.array_equal(full[:1000], part)


@pytest.mark.parametrize("mode", [0, 1, -1, 2])
def test_online_static_walk_equals_offline_and_oracle(orc, mode):
    # mode 0: rows built step by step as walkers reach them; 1: every row first; -1: the library chooses;
    # 2: step by step with the host waiting for the size of every step's row list (option online_device_sized 0)
    from skywalker_amd import capi
    if mode == 2:
        capi.set_option("online_device_sized", 0)
        mode = 0
    xadj, adjncy = orc.rmat_csr(13, 8, 6)
    w = orc.gen_weights(orc.W_UNIFORM, 6, len(adjncy), 1.0, 100.0)
    seeds = orc.gen_seeds(3, 1 << 13, 2000)
    g = capi.Graph.upload(xadj, adjncy, w)
    capi.set_option("online_full_build", mode)
    try:
        p_on, l_on, s_on, _ = g.walk_online(capi.BIAS_STATIC, 1.0, 1.0, seeds, 30, 0.1, 5)
    finally:
        capi.set_option("online_full_build", -1)
        capi.set_option("online_device_sized", 1)
    on = (p_on.to_host((2000, 31)), l_on.to_host())
    g.build_tables()
    p_off, l_off, s_off, _ = g.walk_offline(seeds, 30, 0.1, 5)
    off = (p_off.to_host((2000, 31)), l_off.to_host())
    g.free()
    assert np.array_equal(on[0], off[0]) and np.array_equal(on[1], off[1]) and s_on == s_off
    opaths, olengths, osampled = orc.walk_online(xadj, adjncy, w, 0, 1.0, 1.0, seeds, 30, 0.1, 5)
    assert np.array_equal(on[0], opaths) and np.array_equal(on[1], olengths) and s_on == osampled


@pytest.mark.parametrize("scale,ef,stop", [(11, 8, 0.0), (13, 16, 0.05)])
def test_node2vec_bit_exact(orc, scale, ef, stop):
    from skywalker_amd import capi
    xadj, adjncy = orc.rmat_csr(scale, ef, 31)
    w = orc.gen_weights(orc.W_UNIFORM, 31, len(adjncy), 1.0, 100.0)
    seeds = orc.gen_seeds(2, 1 << scale, 1500)
    g = capi.Graph.upload(xadj, adjncy, w)
    paths, lengths, sampled, _ = g.walk_online(capi.BIAS_NODE2VEC, 2.0, 0.5, seeds, 20, stop, 13)
    got = (paths.to_host((1500, 21)), lengths.to_host())
    g.free()
    opaths, olengths, osampled = orc.walk_online(xadj, adjncy, w, 1, 2.0, 0.5, seeds, 20, stop, 13)
    assert np.array_equal(got[1], olengths)
    assert np.array_equal(got[0], opaths)
    assert sampled == osampled


def test_node2vec_hub_rows_beyond_the_weight_cache(orc):
    # a hub of degree 6000 (more than the kernel keeps in LDS) reached from and returning to small rows
    from skywalker_amd import capi
    rng = np.random.default_rng(12)
    V = 6001
    hub = np.arange(1, V, dtype=np.uint32)
    xadj = np.zeros(V + 1, np.uint32)
    xadj[1] = V - 1
    spokes = []
    for v in range(1, V):
        nb = sorted({0, int(rng.integers(1, V)), int(rng.integers(1, V))} - {v})
        spokes.append(nb)
        xadj[v + 1] = xadj[v] + len(nb)
    adjncy = np.concatenate([hub] + [np.array(s, np.uint32) for s in spokes])
    w = rng.lognormal(0, 1, len(adjncy)).astype(np.float32)
    seeds = rng.integers(0, V, 600, dtype=np.uint32)
    g = capi.Graph.upload(xadj, adjncy, w)
    paths, lengths, sampled, _ = g.walk_online(capi.BIAS_NODE2VEC, 2.0, 0.5, seeds, 12, 0.0, 4)
    got = (paths.to_host((600, 13)), lengths.to_host())
    g.free()
    opaths, olengths, osampled = orc.walk_online(xadj, adjncy, w, 1, 2.0, 0.5, seeds, 12, 0.0, 4)
    assert np.array_equal(got[0], opaths) and np.array_equal(got[1], olengths) and sampled == osampled


@pytest.mark.parametrize("scale,ef,stop,p,q", [(11, 8, 0.0, 2.0, 0.5), (13, 16, 0.05, 0.25, 4.0), (12, 8, 0.0, 1.0, 1.0)])
def test_node2vec_rejection_bit_exact(orc, scale, ef, stop, p, q):
    from skywalker_amd import capi
    xadj, adjncy = orc.rmat_csr(scale, ef, 33)
    w = orc.gen_weights(orc.W_LOGNORMAL, 33, len(adjncy), 0.0, 1.0)
    seeds = orc.gen_seeds(3, 1 << scale, 5000)
    g = capi.Graph.upload(xadj, adjncy, w)
    # no tables yet: the call builds the first-order tables itself
    paths, lengths, sampled, _ = g.walk_online(capi.BIAS_NODE2VEC_REJECT, p, q, seeds, 40, stop, 17)
    got = (paths.to_host((5000, 41)), lengths.to_host())
    prob, alias, valid = g.tables()
    g.free()
    oprob, oalias, ovalid = orc.alias_build(xadj, w)
    assert np.array_equal(prob.view(np.uint32), oprob.view(np.uint32)) and np.array_equal(alias, oalias)
    opaths, olengths, osampled = orc.walk_node2vec_reject(xadj, adjncy, oprob, oalias, p, q, seeds, 40, stop, 17)
    assert np.array_equal(got[1], olengths)
    assert np.array_equal(got[0], opaths)
    assert sampled == osampled


@pytest.mark.parametrize("walkers", [1, 700, 10000, 15000, 40000, 60000, 240000])
@pytest.mark.parametrize("p,q", [(0.25, 1.0), (0.5, 2.0), (0.5, 1.0), (4.0, 1.0), (1.0, 1.0), (0.0625, 8.0), (8.0, 0.0625)])
def test_node2vec_trials_by_how_many_are_kept(orc, walkers, p, q):
    # one trial a turn or four, with 64 lanes a walker to 2; q = 1: no trial needs the previous row; p = q = 1: the first-order walk
    from skywalker_amd import capi
    xadj, adjncy = orc.rmat_csr(11, 12, 35)
    w = orc.gen_weights(orc.W_LOGNORMAL, 35, len(adjncy), 0.0, 2.0)
    w[xadj[3]:xadj[9]] = 0.0  # rows without weight
    prob, alias, _ = orc.alias_build(xadj, w)
    seeds = orc.gen_seeds(6, (1 << 11) + 1, walkers)
    g = capi.Graph.upload(xadj, adjncy, w)
    for stop, length in ((0.0, 7), (0.05, 12)):
        paths, lengths, sampled, _ = g.walk_online(capi.BIAS_NODE2VEC_REJECT, p, q, seeds, length, stop, 19)
        want = orc.walk_node2vec_reject(xadj, adjncy, prob, alias, p, q, seeds, length, stop, 19)
        assert np.array_equal(lengths.to_host(), want[1]) and np.array_equal(paths.to_host((walkers, length + 1)), want[0])
        assert sampled == want[2]
    g.free()


@pytest.mark.parametrize("walkers", [1, 700, 7168, 7169, 14337, 28673, 57344, 57345])
@pytest.mark.parametrize("p,q", [(0.25, 1.0), (0.5, 2.0), (0.0625, 8.0), (2.0, 0.5), (1.0, 1.0)])
def test_node2vec_rejection_on_an_uploaded_table_whose_rows_without_weight_keep_some_columns(orc, walkers, p, q):
    # sky_alias_upload takes any prob in [0, 1] in a row flagged invalid: a trial that keeps its column goes on from there, and
    # the first one that does not ends the walk if no earlier trial of its step was kept; one trial a turn and four, 64 lanes a walker to 4
    from skywalker_amd import capi
    rng = np.random.default_rng(17)
    xadj, adjncy = orc.rmat_csr(11, 12, 35)
    w = orc.gen_weights(orc.W_LOGNORMAL, 35, len(adjncy), 0.0, 2.0)
    V = len(xadj) - 1
    for v in np.flatnonzero(rng.random(V) < 0.3):
        w[xadj[v]:xadj[v + 1]] = 0.0
    prob, alias, valid = orc.alias_build(xadj, w)
    free = alias == 0xFFFFFFFF
    assert free.sum() > len(w) // 8
    prob[free] = rng.choice(np.float32([0.0, 0.3, 0.7, 0.95, 1.0]), free.sum())
    seeds = orc.gen_seeds(6, V + 1, walkers)
    g = capi.Graph.upload(xadj, adjncy, w)
    g.upload_tables(prob, alias, valid)
    for stop, length in ((0.0, 12), (0.02, 30)):
        paths, lengths, sampled, _ = g.walk_online(capi.BIAS_NODE2VEC_REJECT, p, q, seeds, length, stop, 19)
        want = orc.walk_node2vec_reject(xadj, adjncy, prob, alias, p, q, seeds, length, stop, 19)
        assert np.array_equal(lengths.to_host(), want[1]) and np.array_equal(paths.to_host((walkers, length + 1)), want[0])
        assert sampled == want[2]
    g.free()


def test_read_once_gathers_give_the_same_paths(orc):
    from skywalker_amd import capi
    xadj, adjncy = orc.rmat_csr(12, 16, 36)
    w = orc.gen_weights(orc.W_LOGNORMAL, 36, len(adjncy), 0.0, 1.0)
    seeds = orc.gen_seeds(9, 1 << 12, 3000)
    g = capi.Graph.upload(xadj, adjncy, w)
    g.build_tables()
    prob, alias, _ = g.tables()
    want = orc.walk_offline(xadj, adjncy, prob, alias, seeds, 30, 0.02, 21)
    try:
        for mode in (0, 1):
            for indexed in (False, True):
                capi.set_option("walk_read_once", mode)
                g.build_tables()
                if indexed:
                    g.build_walk_index()
                paths, lengths, sampled, _ = g.walk_offline(seeds, 30, 0.02, 21)
                assert np.array_equal(paths.to_host((3000, 31)), want[0]) and np.array_equal(lengths.to_host(), want[1])
                assert sampled == want[2]
        with pytest.raises(capi.SkyError):
            capi.set_option("walk_read_once", 2)
    finally:
        capi.set_option("walk_read_once", -1)
        g.free()


def test_node2vec_rejection_of_large_batches(orc):
    # 300,000 walkers take two lanes each, 70,000 of them four: the paths do not depend on it
    from skywalker_amd import capi
    xadj, adjncy = orc.rmat_csr(12, 16, 35)
    w = orc.gen_weights(orc.W_LOGNORMAL, 35, len(adjncy), 0.0, 1.0)
    seeds = orc.gen_seeds(8, 1 << 12, 300000)
    g = capi.Graph.upload(xadj, adjncy, w)
    g.build_tables()
    paths, lengths, sampled, _ = g.walk_online(capi.BIAS_NODE2VEC_REJECT, 2.0, 0.5, seeds, 10, 0.0, 19)
    big = (paths.to_host((300000, 11)), lengths.to_host())
    small, _, _, _ = g.walk_online(capi.BIAS_NODE2VEC_REJECT, 2.0, 0.5, seeds[:70000], 10, 0.0, 19)
    small = small.to_host((70000, 11))
    prob, alias, valid = g.tables()
    g.free()
    opaths, olengths, osampled = orc.walk_node2vec_reject(xadj, adjncy, prob, alias, 2.0, 0.5, seeds, 10, 0.0, 19)
    assert np.array_equal(big[0], opaths) and np.array_equal(big[1], olengths) and sampled == osampled
    assert np.array_equal(small, opaths[:70000])


@pytest.mark.parametrize("walkers", [1, 7168, 7169, 14337, 28673, 57345, 114689])
def test_node2vec_rejection_group_sizes(orc, walkers):
    # 64, 64, 32, 16, 8, 4 and 2 lanes per walker; rows around the lengths one and two rounds of probes cover, many trials
    from skywalker_amd import capi
    rng = np.random.default_rng(44)
    degs = [0, 1, 2, 3, 4, 5, 7, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65, 79, 80, 81, 287, 1055, 1056, 4159, 4160, 4161] * 12
    xadj, adjncy, w = graph_from_degrees(degs, rng, "sparse")
    seeds = rng.integers(0, len(degs), walkers, dtype=np.uint32)
    g = capi.Graph.upload(xadj, adjncy, w)
    g.build_tables()
    prob, alias, _ = g.tables()
    for p, q, stop in ((0.25, 4.0, 0.02), (4.0, 0.5, 0.0)):
        paths, lengths, sampled, _ = g.walk_online(capi.BIAS_NODE2VEC_REJECT, p, q, seeds, 9, stop, 23)
        want = orc.walk_node2vec_reject(xadj, adjncy, prob, alias, p, q, seeds, 9, stop, 23)
        assert np.array_equal(paths.to_host((walkers, 10)), want[0]) and np.array_equal(lengths.to_host(), want[1])
        assert sampled == want[2]
    g.free()


def test_node2vec_rejection_second_step_law(orc):
    # exact second-order law on a small graph, sampled on the device
    from skywalker_amd import capi
    edges = [(0, 1), (0, 2), (1, 2), (2, 3), (2, 4)]
    wts = [1.0, 2.0, 3.0, 4.0, 5.0]
    src = [a for a, b in edges] + [b for a, b in edges]
    dst = [b for a, b in edges] + [a for a, b in edges]
    ww = wts + wts
    order = np.lexsort((dst, src))
    adjncy = np.array(dst, np.uint32)[order]
    w = np.array(ww, np.float32)[order]
    xadj = np.zeros(6, np.uint32)
    np.add.at(xadj, np.array(src)[order] + 1, 1)
    xadj = np.cumsum(xadj).astype(np.uint32)
    p, q, N = 2.0, 0.5, 400000
    g = capi.Graph.upload(xadj, adjncy, w)
    paths, lengths, sampled, _ = g.walk_online(capi.BIAS_NODE2VEC_REJECT, p, q, np.zeros(N, np.uint32), 2, 0.0, 9)
    paths = paths.to_host((N, 3))
    g.free()
    sel = paths[:, 1] == 2
    second = np.bincount(paths[sel, 2], minlength=5)
    law = np.array([2.0 / p, 3.0, 0.0, 4.0 / q, 5.0 / q])
    law /= law.sum()
    assert second[2] == 0 and sampled == 2 * N
    assert chi_square_p(second[[0, 1, 3, 4]], law[[0, 1, 3, 4]]) > 0.01


def test_start_vertices_that_do_not_exist_never_move(orc):
    # same rule as the oracle's, in every walk kernel: the seed is recorded, the length is 0
    from skywalker_amd import capi
    xadj, adjncy = orc.rmat_csr(10, 8, 3)
    V = len(xadj) - 1
    w = orc.gen_weights(orc.W_UNIFORM, 3, len(adjncy), 1.0, 10.0)
    seeds = orc.gen_seeds(2, V, 300)
    seeds[::7] = V
    seeds[3::11] = 0xFFFFFFFF
    seeds[5] = V + 1

    def host(r, length):
        out = (r[0].to_host((len(seeds), length + 1)), r[1].to_host(), r[2])
        r[0].free()
        r[1].free()
        return out

    g = capi.Graph.upload(xadj, adjncy, w)
    capi.set_option("online_full_build", 0)
    try:
        lazy = host(g.walk_online(capi.BIAS_STATIC, 1.0, 1.0, seeds, 12, 0.05, 9), 12)
    finally:
        capi.set_option("online_full_build", -1)
    n2v = host(g.walk_online(capi.BIAS_NODE2VEC, 2.0, 0.5, seeds, 12, 0.05, 9), 12)
    g.build_tables()
    prob, alias, _ = g.tables()
    off = host(g.walk_offline(seeds, 12, 0.05, 9), 12)
    rej = host(g.walk_online(capi.BIAS_NODE2VEC_REJECT, 2.0, 0.5, seeds, 12, 0.05, 9), 12)
    g.free()
    want = orc.walk_offline(xadj, adjncy, prob, alias, seeds, 12, 0.05, 9)
    for got in (off, lazy):
        assert np.array_equal(got[1], want[1]) and np.array_equal(got[0], want[0]) and got[2] == want[2]
    want = orc.walk_online(xadj, adjncy, w, 1, 2.0, 0.5, seeds, 12, 0.05, 9)
    assert np.array_equal(n2v[1], want[1]) and np.array_equal(n2v[0], want[0]) and n2v[2] == want[2]
    want = orc.walk_node2vec_reject(xadj, adjncy, prob, alias, 2.0, 0.5, seeds, 12, 0.05, 9)
    assert np.array_equal(rej[1], want[1]) and np.array_equal(rej[0], want[0]) and rej[2] == want[2]
    assert np.all(off[1][seeds >= V] == 0)


@pytest.mark.parametrize("every", [0, 1, 7, 16])
@pytest.mark.parametrize("indexed", [False, True])
def test_walk_index_and_walker_lists_give_the_same_paths(orc, indexed, every):
    # the 16-byte walk index and the hand-over of live walkers between launches change how a walk is run, not what
    # it finds: DeepWalk and PPR paths, lengths and counts equal the oracle's
    from skywalker_amd import capi
    xadj, adjncy = orc.rmat_csr(14, 8, 17)
    w = orc.gen_weights(orc.W_LOGNORMAL, 17, len(adjncy), 0.0, 2.0)
    w[xadj[5]:xadj[6]] = 0.0  # a row without weight: walkers that reach it stop there
    V = len(xadj) - 1
    seeds = orc.gen_seeds(4, V, 20011)
    seeds[3] = V + 7
    g = capi.Graph.upload(xadj, adjncy, w)
    g.build_tables()
    prob, alias, _ = g.tables()
    if indexed:
        g.build_walk_index()
    capi.set_option("walk_compact_every", every)
    try:
        for length, stop, seed in ((80, 0.0, 5), (100, 0.15, 6), (3, 0.0, 7)):
            paths, lengths, sampled, _ = g.walk_offline(seeds, length, stop, seed)
            opaths, olengths, osampled = orc.walk_offline(xadj, adjncy, prob, alias, seeds, length, stop, seed)
            assert np.array_equal(lengths.to_host(), olengths)
            assert np.array_equal(paths.to_host((len(seeds), length + 1)), opaths)
            assert sampled == osampled
    finally:
        capi.set_option("walk_compact_every", 0)
    g.free()


def test_walk_index_goes_stale_when_tables_change(orc):
    # the index is a copy of table entries: a rebuild with other weights must not be walked with the old copy
    from skywalker_amd import capi
    xadj, adjncy = orc.rmat_csr(12, 8, 19)
    w1 = orc.gen_weights(orc.W_UNIFORM, 19, len(adjncy), 1.0, 100.0)
    w2 = orc.gen_weights(orc.W_LOGNORMAL, 20, len(adjncy), 0.0, 2.0)
    seeds = orc.gen_seeds(5, len(xadj) - 1, 3000)
    g = capi.Graph.upload(xadj, adjncy, w1)
    g.build_tables()
    g.build_walk_index()
    p2, a2, v2 = orc.alias_build(xadj, w2)
    g.upload_tables(p2, a2, v2)
    paths, lengths, sampled, _ = g.walk_offline(seeds, 30, 0.0, 2)
    opaths, olengths, osampled = orc.walk_offline(xadj, adjncy, p2, a2, seeds, 30, 0.0, 2)
    assert np.array_equal(paths.to_host((3000, 31)), opaths) and sampled == osampled
    g.build_walk_index()
    paths, lengths, sampled, _ = g.walk_offline(seeds, 30, 0.0, 2)
    assert np.array_equal(paths.to_host((3000, 31)), opaths) and sampled == osampled
    g.free()


@pytest.mark.parametrize("dist", ["lognormal2", "nearequal", "sparse"])
@pytest.mark.parametrize("walkers", [1, 256, 257, 4096, 4097])
def test_online_static_draws_evaluated_from_the_weights(orc, walkers, dist):
    # workgroups of 1024 threads to 256; rows around a chunk of 256 slots, and rows of more than 256 chunks; no row with a table, and those
    # that the walk is expected to gain by
    from skywalker_amd import capi
    rng = np.random.default_rng(45)
    degs = [1, 2, 3, 4, 5, 63, 64, 65, 255, 256, 257, 511, 513, 1023, 1025, 4097, 65535, 65536, 65537, 140001, 0] + \
        list(rng.integers(1, 400, 60))
    xadj, adjncy, w = graph_from_degrees(degs, rng, dist)
    seeds = ((np.arange(walkers) + 19) % len(degs)).astype(np.uint32)
    g = capi.Graph.upload(xadj, adjncy, w)
    g.set_option("online_full_build", 0)
    for length, stop in ((1, 0.0), (9, 0.03)):
        want = orc.walk_online(xadj, adjncy, w, 0, 1.0, 1.0, seeds, length, stop, 29)
        for mode in (1, -1):
            g.set_option("online_direct", mode)
            paths, lengths, sampled, _ = g.walk_online(capi.BIAS_STATIC, 1.0, 1.0, seeds, length, stop, 29)
            assert np.array_equal(lengths.to_host(), want[1]) and np.array_equal(paths.to_host((walkers, length + 1)), want[0])
            assert sampled == want[2]
    g.free()


@pytest.mark.parametrize("walkers", [512, 513, 1025])
def test_node2vec_table_rows_beyond_the_window(orc, walkers):
    # eight and four wavefronts per walker, windows of 1024 and 512 ids; rows of more than 65,536 entries (membership is searched again instead of kept),
    # previous rows of many windows, and of more than 32 times the current row's length
    from skywalker_amd import capi
    rng = np.random.default_rng(46)
    degs = list(rng.integers(0, 300, 1500)) + list(rng.integers(900, 4200, 250)) + [1023, 1024, 1025] * 30 + \
        list(rng.integers(20000, 65537, 30)) + [65537, 66001, 140003] * 6
    rng.shuffle(degs)
    xadj, adjncy, w = graph_from_degrees(degs, rng, "sparse", V=len(degs) + 3)
    rows = np.argsort(np.diff(xadj))[-400:]
    seeds = rng.choice(rows, walkers).astype(np.uint32)
    g = capi.Graph.upload(xadj, adjncy, w)
    paths, lengths, sampled, _ = g.walk_online(capi.BIAS_NODE2VEC, 4.0, 0.25, seeds, 7, 0.0, 31)
    want = orc.walk_online(xadj, adjncy, w, 1, 4.0, 0.25, seeds, 7, 0.0, 31)
    assert np.array_equal(lengths.to_host(), want[1]) and np.array_equal(paths.to_host((walkers, 8)), want[0])
    assert sampled == want[2]
    g.free()


@pytest.mark.parametrize("V", [1200, (1 << 18) - 1, 1 << 18, (1 << 18) + 1])
@pytest.mark.parametrize("walkers,p,q", [(768, 2.0, 0.5), (769, 3.0, 0.7), (2000, 0.25, 4.0)])
def test_node2vec_table_with_a_bit_per_vertex(orc, V, walkers, p, q):
    # eight and four wavefronts per walker, the largest graph whose vertices have bits and the first without; quotients by powers of two
    # and by others; rows around the 4 and 16 slots a thread of the draw and around the weights kept; previous rows of more than
    # 32,768 entries before short ones (searched in memory) and long ones; surpluses beyond 64 bits
    from skywalker_amd import capi
    rng = np.random.default_rng(47)
    degs = [1, 2, 3, 4, 5, 987, 988, 989, 1023, 1024, 1025, 2047, 2048, 2049, 4095, 4096, 4097, 8191, 8192, 8193] * 4 + \
        [32767, 32768, 32769, 40000, 66001] + list(rng.integers(1, 900, 500))
    n = len(degs)
    ids = np.sort(np.append(rng.choice(np.arange(1, V - 1), n - 2, replace=False), [0, V - 1]))  # the vertices with rows
    rng.shuffle(degs)
    lens = np.zeros(V, np.int64)
    lens[ids] = degs
    xadj = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)
    adjncy = np.concatenate([np.sort(rng.choice(ids, k)) for k in degs]).astype(np.uint32)
    w = weights(len(adjncy), rng, "sparse")
    for v in ids[::3]:
        w[xadj[v]:xadj[v + 1]] *= np.float32(1e-19)
    seeds = np.append(rng.choice(ids, walkers - 2), [V - 1, 0]).astype(np.uint32)
    g = capi.Graph.upload(xadj, adjncy, w)
    paths, lengths, sampled, _ = g.walk_online(capi.BIAS_NODE2VEC, p, q, seeds, 8, 0.02, 37)
    got = paths.to_host((walkers, 9)), lengths.to_host()
    g.free()
    want = orc.walk_online(xadj, adjncy, w, 1, p, q, seeds, 8, 0.02, 37)
    assert np.array_equal(got[1], want[1]) and np.array_equal(got[0], want[0])
    assert sampled == want[2]


@pytest.mark.parametrize("kind", ["uniform", "equal", "sparse", "tiny"])
@pytest.mark.parametrize("walkers", [300, 1000])
def test_node2vec_table_rows_of_one_wavefront(orc, walkers, kind):
    # rows around the 256 entries that one wavefront draws from by itself, and around the 4,095 up to which the workgroup holds them; weights that
    # sum up exactly in doubles or not, none lighter than the others, most of no weight, all next to none
    from skywalker_amd import capi
    rng = np.random.default_rng(53)
    degs = list(range(1, 9)) * 4 + [63, 64, 65, 127, 128, 129] * 6 + list(range(250, 262)) * 12 + [4094, 4095, 4096, 4097] * 3
    rng.shuffle(degs)
    n = len(degs)
    xadj = np.concatenate([[0], np.cumsum(degs)]).astype(np.uint32)
    adjncy = np.concatenate([np.sort(rng.integers(0, n, k)) for k in degs]).astype(np.uint32)
    w = weights(len(adjncy), rng, {"tiny": "sparse"}.get(kind, kind))
    if kind == "tiny":
        w *= np.float32(1e-19)
    seeds = rng.integers(0, n, walkers).astype(np.uint32)
    g = capi.Graph.upload(xadj, adjncy, w)
    paths, lengths, sampled, _ = g.walk_online(capi.BIAS_NODE2VEC, 2.0, 0.5, seeds, 10, 0.0, 41)
    got = paths.to_host((walkers, 11)), lengths.to_host()
    g.free()
    want = orc.walk_online(xadj, adjncy, w, 1, 2.0, 0.5, seeds, 10, 0.0, 41)
    assert np.array_equal(got[1], want[1]) and np.array_equal(got[0], want[0])
    assert sampled == want[2]


def nearly_vanishing_row(d, lights):
    """One weight counts in the row's sum, of d; `lights` weigh next to nothing, the others a hair less than what counts: d - 1 shares each."""
    u = 2.0 ** -64
    w = np.full(d, u * (1 - 2.0 ** -24))
    w[d // 3] = u
    w[np.random.default_rng(d).permutation(np.delete(np.arange(d), d // 3))[:lights]] = u * 2.0 ** -30
    return w.astype(np.float32)


@pytest.mark.parametrize("walkers", [300, 1000, 3000, 9000])
def test_draws_from_rows_whose_surpluses_come_close_to_64_bits(orc, walkers):
    # the longest rows that are held, by a wavefront or a workgroup, have sums just below 2^64; longer ones pass it, some by next to nothing, so that
    # what wraps is below the deficits of most lights; walkers of 512, 256, 128 and 64 threads
    from skywalker_amd import capi
    near = [(d, 3) for d in (63, 64, 65, 255, 256, 257, 511, 512, 513, 1024, 1025, 2048, 2049, 4094, 4095, 4096, 4097)]
    past = [(4227, 257), (4361, 513), (7080, 4710), (7941, 5828)]
    rows = [nearly_vanishing_row(d, k) for d, k in near + past]
    for w, (d, k) in zip(rows, near + past):
        surplus = np.maximum(w.astype(np.float64) * 2.0 ** 64 * d - 1, 0).sum()  # the weights' sum is 1; 2^24 of these pass 64 bits
        if (d, k) in past:
            assert 0 < surplus - 2 ** 24 < k / 4
        else:
            assert surplus < 2 ** 24 and (d < 4094 or surplus > 0.998 * 2 ** 24)
    w = np.concatenate(rows + [np.ones(32 * 20000, np.float32)])
    lens = np.concatenate([[len(r) for r in rows], np.full(20000, 32)])
    xadj = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)
    adjncy = np.arange(len(w), dtype=np.uint32) - np.repeat(xadj[:-1], lens)  # a vertex of its own for every slot of a row
    seeds = np.arange(walkers, dtype=np.uint32) % len(rows)
    seeds[walkers // 2:] = len(near) + seeds[walkers // 2:] % len(past)
    oprob, oalias, _ = orc.alias_build(xadj, w)
    want = orc.walk_offline(xadj, adjncy, oprob, oalias, seeds, 1, 0.0, 5)[0].ravel()
    g = capi.Graph.upload(xadj, adjncy, w)
    g.set_option("online_full_build", 0)
    g.set_option("online_direct", 1)  # no row is built
    for bias in (capi.BIAS_STATIC, capi.BIAS_NODE2VEC):
        assert np.array_equal(g.walk_online(bias, 2.0, 0.5, seeds, 1, 0.0, 5)[0].to_host(), want), bias
    g.free()


@pytest.mark.parametrize("kind", ["uniform", "lognormal", "equal", "sparse", "tiny"])
@pytest.mark.parametrize("walkers", [900, 3000, 9000])
def test_online_static_draws_from_short_rows(orc, walkers, kind):
    # walkers of four wavefronts, two and one; rows around the 64 entries that have a slot a lane, the 256 that have four and
    # the 512 that have eight where a walker is one wavefront
    from skywalker_amd import capi
    rng = np.random.default_rng(59)
    degs = list(range(1, 9)) * 4 + [31, 32, 33, 62, 63, 64, 65, 66, 127, 128, 129] * 6 + list(range(252, 260)) * 6 + [300, 509, 510, 511, 512, 513, 1025] * 2
    rng.shuffle(degs)
    n = len(degs)
    xadj = np.concatenate([[0], np.cumsum(degs)]).astype(np.uint32)
    adjncy = np.concatenate([np.sort(rng.integers(0, n, k)) for k in degs]).astype(np.uint32)
    w = weights(len(adjncy), rng, {"tiny": "sparse"}.get(kind, kind))
    if kind == "tiny":
        w *= np.float32(1e-19)
    seeds = rng.integers(0, n, walkers).astype(np.uint32)
    g = capi.Graph.upload(xadj, adjncy, w)
    g.set_option("online_full_build", 0)
    g.set_option("online_direct", 1)
    paths, lengths, sampled, _ = g.walk_online(capi.BIAS_STATIC, 1.0, 1.0, seeds, 12, 0.02, 43)
    got = paths.to_host((walkers, 13)), lengths.to_host()
    g.free()
    want = orc.walk_online(xadj, adjncy, w, 0, 1.0, 1.0, seeds, 12, 0.02, 43)
    assert np.array_equal(got[1], want[1]) and np.array_equal(got[0], want[0])
    assert sampled == want[2]


@pytest.mark.parametrize("longest,walkers", [(70001, 256), (70001, 257), (70001, 8193), (40001, 512), (40001, 513), (40001, 16385),
                                             (12289, 1024), (12289, 1025), (12289, 8193)])
def test_online_static_draws_by_workgroups_of_every_size(longest, walkers):
    # 64 to 1024 threads a walker by the longest row and the number of walkers; rows around 256 slots a wavefront and 4 a thread,
    # none of which is built (online_direct 1), or those that a walk from these vertices is expected to gain by (-1)
    from skywalker_amd import capi
    rng = np.random.default_rng(longest)
    lens = [1, 2, 3, 4, 5, 255, 256, 257, 511, 512, 513, 1023, 1024, 1025, 2047, 2048, 2049, 4095, 4096, 4097, longest] + \
        list(rng.integers(1, 5000, 100))
    n = len(lens)
    lens = np.concatenate([lens, np.full(625000, 32)])
    xadj = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)
    local = np.arange(xadj[-1], dtype=np.uint32) - np.repeat(xadj[:-1], lens)  # a vertex of its own for every slot of a row
    w = np.ones(xadj[-1], np.float32)
    w[:xadj[n]] = weights(int(xadj[n]), rng, "sparse")
    g = capi.Graph.upload(xadj, local, w)
    g.set_option("online_full_build", 0)
    seeds = (np.arange(walkers) % n).astype(np.uint32)
    online = []
    for mode in (1, -1):
        g.set_option("online_direct", mode)
        online.append(g.walk_online(capi.BIAS_STATIC, 1.0, 1.0, seeds, 1, 0.0, 7))
    g.build_tables()
    tabled = g.walk_offline(seeds, 1, 0.0, 7)
    for direct in online:
        assert np.array_equal(direct[0].to_host(), tabled[0].to_host()) and np.array_equal(direct[1].to_host(), tabled[1].to_host())
        assert direct[2] == tabled[2]
    g.free()


def test_node2vec_rejection_without_bias_by_more_walkers_than_one_launch_has():
    # p = q = 1 goes by the first-order walk, whose grid for so many walkers would be empty
    from skywalker_amd import capi
    N = 0xFFFFFF10
    if capi.mem_info()[0] < 14 * N:
        pytest.skip("56 GB of device memory")
    xadj, adjncy = np.array([0, 1, 2], np.uint32), np.array([1, 0], np.uint32)
    g = capi.Graph.upload(xadj, adjncy, np.ones(2, np.float32))
    g.build_tables()
    seeds = capi.DeviceArray(N, np.uint32, fill=1)
    paths, lengths = capi.DeviceArray(N, np.uint32, fill=7), capi.DeviceArray(N, np.uint32, fill=7)
    sampled = g.walk_online(capi.BIAS_NODE2VEC_REJECT, 1.0, 1.0, seeds, 0, 0.0, 5, out=(paths, lengths))[2]
    assert sampled == 0
    import ctypes as C
    for first in (0, (1 << 31) - 500, (1 << 32) - 2000, N - 1000):
        for array, want in ((paths, 1), (lengths, 0)):
            part = np.empty(1000 if first + 1000 <= N else N - first, np.uint32)
            capi._ck(capi.lib().sky_memcpy_d2h(capi._p(part), C.c_void_p(array.ptr.value + 4 * first), C.c_size_t(part.nbytes)))
            assert (part == want).all()
    for x in (seeds, paths, lengths, g):
        x.free()


@pytest.mark.parametrize("full_build", [0, -1])
@pytest.mark.parametrize("length", [1, 2])
def test_short_walks_from_well_connected_vertices_build_their_rows(orc, length, full_build):
    # a walk of a few steps from any vertices needs no tables; from the longest row for every walker it does, and sweeping it
    # for each of them takes ten times as long as the others
    from skywalker_amd import capi
    xadj, adjncy = orc.rmat_csr(16, 16, 44)
    w = orc.gen_weights(orc.W_LOGNORMAL, 44, len(adjncy), 0.0, 1.0)
    deg = np.diff(xadj.astype(np.int64))
    prob, alias, _ = orc.alias_build(xadj, w)
    rng = np.random.default_rng(44)
    N = 40000
    g = capi.Graph.upload(xadj, adjncy, w)
    g.set_option("online_full_build", full_build)
    starts = {"any": rng.integers(0, len(deg) + 1, N), "ends": adjncy[rng.integers(0, len(adjncy), N)], "first": np.arange(N) % 5000,
              "hub": np.full(N, deg.argmax()), "none": np.full(N, len(deg)), "few": np.argsort(-deg)[:7]}
    took = {}
    for name, seeds in starts.items():
        seeds = seeds.astype(np.uint32)
        paths, lengths, sampled = orc.walk_offline(xadj, adjncy, prob, alias, seeds, length, 0.0, 5)
        for _ in range(4):
            got = g.walk_online(capi.BIAS_STATIC, 1.0, 1.0, seeds, length, 0.0, 5)
            took[name] = min(took.get(name, 1e9), got[3])
            assert np.array_equal(got[0].to_host(paths.shape), paths) and np.array_equal(got[1].to_host(), lengths) and got[2] == sampled
            if full_build:
                g.sample_session(np.zeros(0, np.uint32), [1, 2], 1)  # its begin leaves the graph without tables
    print({k: "%.1f us" % (v * 1e6) for k, v in took.items()})
    assert took["hub"] < 3 * took["any"]
    g.free()


@pytest.mark.parametrize("walkers", [32704, 32705, 32768, 32769, 100001])
def test_sampled_edges_counted_in_one_word_and_in_many(orc, walkers):
    # 511 and 512 wavefronts of a walker a lane, which add to one word and to 64, more of them in the rejection walk, counts behind a
    # kernel of their own: one call after another on the same words, each of which starts from zero
    from skywalker_amd import capi
    xadj, adjncy = orc.rmat_csr(12, 8, 77)
    w = orc.gen_weights(orc.W_UNIFORM, 77, len(adjncy), 1.0, 100.0)
    seeds = orc.gen_seeds(3, 1 << 12, walkers)
    g = capi.Graph.upload(xadj, adjncy, w)
    g.set_option("online_full_build", 0)
    runs = [lambda: g.walk_online(capi.BIAS_STATIC, 1.0, 1.0, seeds, 2, 0.0, 5)]
    for _ in range(2):
        runs += [lambda: g.walk_offline(seeds, 6, 0.15, 5), lambda: g.walk_online(capi.BIAS_NODE2VEC_REJECT, 2.0, 0.5, seeds, 4, 0.0, 5),
                 lambda: g.walk_online(capi.BIAS_NODE2VEC_REJECT, 0.25, 1.0, seeds[:700], 4, 0.0, 5), lambda: g.walk_offline(seeds[:100], 6, 0.0, 5)]
    for k, run in enumerate(runs):
        if k == 1:
            g.build_tables()
        _, lengths, sampled, _ = run()
        assert sampled == int(lengths.to_host().sum()) > 0, k
    g.free()


@pytest.mark.parametrize("index", [False, True])
@pytest.mark.parametrize("walkers", [8193, 8207, 8208, 49152, 49153])
def test_walks_of_sixteen_walkers_a_wavefront(orc, walkers, index):
    # tables of more than 32 MB: partly filled wavefronts and workgroups, the most walkers that go sixteen to a wavefront and one more;
    # walkers that end at vertices without edges, at the stop test, alone in their wavefronts, and at a start vertex that does not exist
    from skywalker_amd import capi
    xadj, adjncy = orc.rmat_csr(17, 34, 5)
    w = orc.gen_weights(orc.W_UNIFORM, 5, len(adjncy), 1.0, 100.0)
    seeds = orc.gen_seeds(3, 1 << 17, walkers)
    seeds[-1] = 1 << 17
    g = capi.Graph.upload(xadj, adjncy, w)
    g.build_tables()
    if index:
        g.build_walk_index()
    prob, alias, _ = g.tables()
    for stop in (0.15, 0.0):
        paths, lengths, sampled, _ = g.walk_offline(seeds, 24, stop, 9)
        want = orc.walk_offline(xadj, adjncy, prob, alias, seeds, 24, stop, 9)
        assert np.array_equal(lengths.to_host(), want[1]) and np.array_equal(paths.to_host((walkers, 25)), want[0]) and sampled == want[2]
    g.free()


@pytest.mark.parametrize("streams", [1, 0])
@pytest.mark.parametrize("E", [(1 << 24) - 1, 1 << 24])
def test_online_walks_that_build_the_longer_rows(orc, E, streams):
    # the largest graph whose longer rows are built in order and the smallest where they go out beside one another: rows of two wavefronts and
    # more, merged and held ones, streamed ones, ones by tiles; the third walk finds what the first two left
    from skywalker_amd import capi
    rng = np.random.default_rng(67)
    degs = list(rng.integers(510, 2558, 900)) + list(rng.integers(2558, 5118, 500)) + list(rng.integers(5118, 8190, 200)) + \
        list(rng.integers(8190, 24577, 250)) + list(rng.integers(24577, 65534, 12)) + [70001, 600001] + list(rng.integers(33, 510, 3000))
    left = E - sum(degs)
    degs += [31] * (left // 31) + [left % 31]
    rng.shuffle(degs)
    xadj = np.concatenate([[0], np.cumsum(degs)]).astype(np.uint32)
    V = len(degs)
    adjncy = rng.integers(0, V, E, dtype=np.uint32)
    long_rows = np.flatnonzero(np.array(degs) >= 510)
    some = rng.random(E) < 0.5
    adjncy[some] = rng.choice(long_rows, int(some.sum()))
    w = rng.lognormal(0, 2, E).astype(np.float32)
    seeds = rng.integers(0, V, 6000).astype(np.uint32)
    prob, alias, _ = orc.alias_build(xadj, w)
    want = orc.walk_offline(xadj, adjncy, prob, alias, seeds, 12, 0.0, 5)
    g = capi.Graph.upload(xadj, adjncy, w)
    g.set_option("online_full_build", 0)
    g.set_option("build_streams", streams)
    for _ in range(3):
        paths, lengths, sampled, _ = g.walk_online(capi.BIAS_STATIC, 1.0, 1.0, seeds, 12, 0.0, 5)
        assert np.array_equal(lengths.to_host(), want[1]) and np.array_equal(paths.to_host(want[0].shape), want[0]) and sampled == want[2]
    g.free()
