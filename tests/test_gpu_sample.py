"""k-hop neighbour sampling on the GPU against the oracle: bit-exact blocks and counts."""
import numpy as np
import pytest

from helpers import chi_square_p, graph_from_degrees, weights

pytestmark = pytest.mark.gpu


def test_layout_closed_form():
    from skywalker_amd import capi
    assert capi.sample_layout([1, 25, 10]) == (276, 26)
    assert capi.sample_layout([1, 2, 2]) == (7, 3)
    assert capi.sample_layout([1, 20, 20]) == (421, 21)


@pytest.mark.parametrize("device_sized,direct", [(1, 0), (1, -1), (0, -1)])
@pytest.mark.parametrize("fanout", [[1, 25, 10], [1, 3, 2, 2], [1, 5]])
def test_offline_and_online_match_oracle(orc, fanout, device_sized, direct):
    # device_sized 1 (the default): the size of every frontier stays on the device and the host never waits inside
    # the call, or, where the first hop is drawn from the weights (direct), once behind that; 0: the host reads it before it launches the
    # build of the frontier's rows
    from skywalker_amd import capi
    xadj, adjncy = orc.rmat_csr(13, 8, 21)
    w = orc.gen_weights(orc.W_LOGNORMAL, 21, len(adjncy), 0.0, 1.0)
    seeds = orc.gen_seeds(4, 1 << 13, 1500)
    lps, slen = capi.sample_layout(fanout)
    g = capi.Graph.upload(xadj, adjncy, w)
    capi.set_option("online_device_sized", device_sized)
    g.set_option("online_direct", direct)
    try:
        d_on, sl_on, s_on, _ = g.sample_online(seeds, fanout, 17)
    finally:
        capi.set_option("online_device_sized", 1)
    on = (d_on.to_host((1500, lps)), sl_on.to_host((1500, slen)))
    g.build_tables()
    prob, alias, valid = g.tables()
    d_off, sl_off, s_off, _ = g.sample_offline(seeds, fanout, 17)
    off = (d_off.to_host((1500, lps)), sl_off.to_host((1500, slen)))
    g.free()
    odata, osl, osampled = orc.sample_offline(xadj, adjncy, prob, alias, seeds, fanout, 17)
    assert np.array_equal(off[1], osl) and np.array_equal(off[0], odata) and s_off == osampled
    assert np.array_equal(on[0], off[0]) and np.array_equal(on[1], off[1]) and s_on == s_off
    o2data, o2sl, o2sampled = orc.sample_online(xadj, adjncy, w, seeds, fanout, 17)
    assert np.array_equal(on[0], o2data) and np.array_equal(on[1], o2sl) and s_on == o2sampled
    assert osampled == int(osl.sum())


@pytest.mark.parametrize("fanout", [[1, 25, 10], [1, 3, 2, 2], [1, 64]])
def test_distinct_children_match_oracle(orc, fanout):
    # option sample_distinct: the reference's online rule (no slot of a row twice, at most 11 tries per draw)
    from skywalker_amd import capi
    xadj, adjncy = orc.rmat_csr(13, 8, 22)
    w = orc.gen_weights(orc.W_LOGNORMAL, 22, len(adjncy), 0.0, 2.0)  # skewed rows: tries do run out
    seeds = orc.gen_seeds(5, 1 << 13, 1500)
    lps, slen = capi.sample_layout(fanout)
    g = capi.Graph.upload(xadj, adjncy, w)
    capi.set_option("sample_distinct", 1)
    try:
        d_on, sl_on, s_on, _ = g.sample_online(seeds, fanout, 23)
        on = (d_on.to_host((1500, lps)), sl_on.to_host((1500, slen)))
        g.build_tables()
        d_off, sl_off, s_off, _ = g.sample_offline(seeds, fanout, 23)
        off = (d_off.to_host((1500, lps)), sl_off.to_host((1500, slen)))
        with pytest.raises(capi.SkyError):
            g.sample_offline(seeds, [1, 65], 23)
    finally:
        capi.set_option("sample_distinct", 0)
    prob, alias, valid = g.tables()
    g.free()
    odata, osl, osampled = orc.sample_offline(xadj, adjncy, prob, alias, seeds, fanout, 23, distinct=True)
    assert np.array_equal(off[1], osl) and np.array_equal(off[0], odata) and s_off == osampled
    assert np.array_equal(on[0], off[0]) and np.array_equal(on[1], off[1]) and s_on == s_off
    assert osampled == int(osl.sum())
    if fanout[1] >= 25:
        deg = np.diff(xadj)
        big = deg[seeds] > fanout[1]
        assert (osl[big, 0] < fanout[1]).any()  # a parent that ended with fewer children than its fanout is among the cases


@pytest.mark.parametrize("weights", ["lognormal2", "sparse"])
@pytest.mark.parametrize("fanout", [[1, 1, 2], [1, 3, 5], [1, 9, 16], [1, 17, 2], [1, 33, 1], [1, 63], [1, 64]])
def test_distinct_children_of_rows_held_in_lds(orc, fanout, weights):
    # a group of lanes holds a row of at most four entries a lane, and of at most 64, and finds taken slots by their bits: rows
    # at both limits and at the fan-out's, with draws that run out of tries (a few entries with most of the weight)
    from skywalker_amd import capi
    rng = np.random.default_rng(61)
    degs = [0, 1, 2, 3, 4, 5, 15, 16, 17, 18, 31, 32, 33, 34, 35, 62, 63, 64, 65, 66, 130]
    xadj, adjncy, w = graph_from_degrees(degs * 12, rng, weights)
    V = len(xadj) - 1
    prob, alias, valid = orc.alias_build(xadj, w)
    seeds = rng.integers(0, V + 1, 700).astype(np.uint32)
    lps, slen = capi.sample_layout(fanout)
    want = orc.sample_offline(xadj, adjncy, prob, alias, seeds, fanout, 29, distinct=True)
    g = capi.Graph.upload(xadj, adjncy, w)
    g.build_tables()
    g.set_option("sample_distinct", 1)
    for call in (g.sample_offline, g.sample_online):
        data, sl, sampled, _ = call(seeds, fanout, 29)
        assert np.array_equal(sl.to_host((700, slen)), want[1]) and np.array_equal(data.to_host((700, lps)), want[0])
        assert sampled == want[2]
    g.free()


@pytest.mark.parametrize("weights", ["lognormal", "equal", "sparse", "tiny"])
@pytest.mark.parametrize("fanout", [[1, 3], [1, 20, 2], [1, 63], [1, 70]])
def test_online_children_of_short_rows_from_the_weights(orc, fanout, weights):
    # rows around the 64 entries that have a slot a lane, longer than the fan-out and not (those are taken whole); a draw for all lanes but one, and
    # fan-outs that only longer rows draw for; weights that sum up exactly in doubles or not, most of none, all next to none
    from skywalker_amd import capi
    rng = np.random.default_rng(71)
    degs = [0, 1, 2, 3, 4, 5, 19, 20, 21, 22, 31, 32, 33, 62, 63, 64, 65, 66, 69, 70, 71, 130]
    xadj, adjncy, w = graph_from_degrees(degs * 12, rng, {"tiny": "sparse"}.get(weights, weights))
    if weights == "tiny":
        w = w * np.float32(1e-19)
    seeds = rng.integers(0, len(xadj), 700).astype(np.uint32)
    lps, slen = capi.sample_layout(fanout)
    want = orc.sample_online(xadj, adjncy, w, seeds, fanout, 31)
    g = capi.Graph.upload(xadj, adjncy, w)
    g.set_option("online_direct", 1)
    data, sl, sampled, _ = g.sample_online(seeds, fanout, 31)
    assert np.array_equal(sl.to_host((700, slen)), want[1]) and np.array_equal(data.to_host((700, lps)), want[0])
    assert sampled == want[2]
    g.free()


def test_online_sampling_with_short_rows_built_in_vertex_order(orc):
    # option small_in_place = 1 on a list of frontier vertices (by default only builds of 2^25 rows and more use it)
    from skywalker_amd import capi
    xadj, adjncy = orc.rmat_csr(13, 8, 24)
    w = orc.gen_weights(orc.W_LOGNORMAL, 24, len(adjncy), 0.0, 1.0)
    seeds = orc.gen_seeds(6, 1 << 13, 1200)
    fanout = [1, 6, 4, 3]
    lps, slen = capi.sample_layout(fanout)
    g = capi.Graph.upload(xadj, adjncy, w)
    capi.set_option("small_in_place", 1)
    try:
        d_on, sl_on, s_on, _ = g.sample_online(seeds, fanout, 29)
        with pytest.raises(capi.SkyError):
            capi.set_option("small_in_place", 2)
    finally:
        capi.set_option("small_in_place", -1)
    got = (d_on.to_host((1200, lps)), sl_on.to_host((1200, slen)))
    g.free()
    odata, osl, osampled = orc.sample_online(xadj, adjncy, w, seeds, fanout, 29)
    assert np.array_equal(got[0], odata) and np.array_equal(got[1], osl) and s_on == osampled


def test_exact_count_when_every_degree_exceeds_fanout(orc):
    from skywalker_amd import capi
    rng = np.random.default_rng(6)
    V = 500
    xadj, adjncy, w = graph_from_degrees(rng.integers(30, 60, V), rng, "uniform", V=V)
    g = capi.Graph.upload(xadj, adjncy, w)
    g.build_tables()
    seeds = rng.integers(0, V, 300, dtype=np.uint32)
    data, sl, sampled, _ = g.sample_offline(seeds, [1, 25, 10], 3)
    g.free()
    assert sampled == 300 * (25 + 250)
    assert not np.any(data.to_host() == 0xFFFFFFFF)


def test_per_parent_draw_frequencies(orc):
    from skywalker_amd import capi
    rng = np.random.default_rng(9)
    d = 40
    xadj = np.zeros(d + 2, np.uint32)
    xadj[1:] = d
    adjncy = np.arange(1, d + 1, dtype=np.uint32)
    w = rng.lognormal(0, 1, d).astype(np.float32)
    g = capi.Graph.upload(xadj, adjncy, w)
    g.build_tables()
    N = 20000
    data, sl, sampled, _ = g.sample_offline(np.zeros(N, np.uint32), [1, 10], 5)
    g.free()
    draws = data.to_host((N, 11))[:, 1:].ravel()
    assert sampled == N * 10
    assert chi_square_p(np.bincount(draws, minlength=d + 1)[1:], w.astype(np.float64) / w.sum(dtype=np.float64)) > 0.01


def test_seeds_that_do_not_exist_have_no_children(orc):
    from skywalker_amd import capi
    xadj, adjncy = orc.rmat_csr(10, 8, 5)
    V = len(xadj) - 1
    w = orc.gen_weights(orc.W_UNIFORM, 5, len(adjncy), 1.0, 10.0)
    seeds = orc.gen_seeds(6, V, 200)
    seeds[::5] = V
    seeds[1] = 0xFFFFFFFF
    fanout = [1, 4, 3]
    lps, slen = capi.sample_layout(fanout)
    g = capi.Graph.upload(xadj, adjncy, w)
    d_on, sl_on, s_on, _ = g.sample_online(seeds, fanout, 3)
    on = (d_on.to_host((200, lps)), sl_on.to_host((200, slen)))
    g.build_tables()
    d_off, sl_off, s_off, _ = g.sample_offline(seeds, fanout, 3)
    off = (d_off.to_host((200, lps)), sl_off.to_host((200, slen)))
    g.free()
    odata, osl, osampled = orc.sample_online(xadj, adjncy, w, seeds, fanout, 3)
    for got, s in ((on, s_on), (off, s_off)):
        assert np.array_equal(got[0], odata) and np.array_equal(got[1], osl) and s == osampled
    assert np.all(osl[seeds >= V] == 0)


def test_online_sampling_builds_rows_of_every_class_without_waiting(orc):
    # frontiers whose rows fall into every degree class up to the streaming kernel's, their sizes known to the
    # device alone; a second call on the same graph finds the row lists in place
    from helpers import graph_from_degrees
    from skywalker_amd import capi
    rng = np.random.default_rng(77)
    degs = [0, 1, 2, 3, 8, 9, 16, 17, 32, 33, 64, 65, 128, 129, 160, 161, 192, 193, 253, 254, 509, 510, 1021, 1022]
    degs += [512 * nw - 3 for nw in range(3, 11)] + [5118, 6500, 8190, 9000, 25000, 70000, 300000]
    degs += list(rng.integers(0, 300, 600))
    rng.shuffle(degs)
    xadj, adjncy, w = graph_from_degrees(degs, rng, "lognormal")
    V = len(xadj) - 1
    fanout = [1, 4, 3]
    lps, slen = capi.sample_layout(fanout)
    g = capi.Graph.upload(xadj, adjncy, w)
    for rep, (n, mode) in enumerate(((V, 0), (50, 0), (V, -1), (50, -1))):
        g.set_option("online_direct", mode)
        seeds = np.arange(n, dtype=np.uint32) if n == V else rng.integers(0, V, n).astype(np.uint32)
        d_on, sl_on, s_on, _ = g.sample_online(seeds, fanout, 31 + rep)
        odata, osl, osampled = orc.sample_online(xadj, adjncy, w, seeds, fanout, 31 + rep)
        assert np.array_equal(d_on.to_host((n, lps)), odata) and np.array_equal(sl_on.to_host((n, slen)), osl)
        assert s_on == osampled
    g.free()


def test_sampling_hop_by_hop_with_the_callers_weights(orc):
    # sky_sample_session_*: the frontier of every hop is handed out, the rows are built from the weights the caller
    # gives for that hop.  With the graph's own weights the result is sky_sample_online's; with other weights it is
    # the oracle's online sample on a graph that carries those
    from skywalker_amd import capi
    xadj, adjncy = orc.rmat_csr(12, 8, 23)
    w = orc.gen_weights(orc.W_LOGNORMAL, 23, len(adjncy), 0.0, 1.0)
    w2 = orc.gen_weights(orc.W_UNIFORM, 29, len(adjncy), 1.0, 100.0)
    seeds = orc.gen_seeds(6, 1 << 12, 900)
    fanout = [1, 6, 4]
    lps, slen = capi.sample_layout(fanout)
    g = capi.Graph.upload(xadj, adjncy, w)
    d0, s0, n0, _ = g.sample_online(seeds, fanout, 31)
    want = (d0.to_host((900, lps)), s0.to_host((900, slen)), n0)
    d1, s1, n1, _ = g.sample_session(seeds, fanout, 31)
    assert np.array_equal(d1.to_host((900, lps)), want[0]) and np.array_equal(s1.to_host((900, slen)), want[1]) and n1 == n0
    import ctypes
    E = len(w2)
    w2_d = capi.DeviceArray.from_host(w2)
    # the same weights in memory that ends with the last of them (the allocation holds 4 * (E + 8) + 16 bytes): the
    # library copies such an array before its kernels read whole vectors from it
    room = capi.DeviceArray(E + 8, np.float32)

    class Exact:
        ptr = ctypes.c_void_p(room.ptr.value + 32)
    capi._ck(capi.lib().sky_memcpy_h2d(Exact.ptr, capi._p(w2), E * 4))
    odata, osl, osampled = orc.sample_online(xadj, adjncy, w2, seeds, fanout, 31)
    for arr in (w2_d, Exact):
        uppers = []
        d2, s2, n2, _ = g.sample_session(seeds, fanout, 31, lambda hop, upper: (uppers.append(upper), arr)[1])
        got = (d2.to_host((900, lps)), s2.to_host((900, slen)))
        assert uppers[0] == 900 and 0 < uppers[1] <= 900 * 6
        assert np.array_equal(got[1], osl) and np.array_equal(got[0], odata) and n2 == osampled
    g.free()


@pytest.mark.parametrize("distinct", [False, True])
@pytest.mark.parametrize("n,fanout", [(3, [1, 64, 5]), (4095, [1, 1, 2, 17]), (4096, [1, 33, 3]), (9000, [1, 3, 1, 4, 2]),
                                      (70001, [1, 7, 4])])
def test_batches_by_workgroup_and_by_hop(orc, n, fanout, distinct):
    # few start vertices share workgroups hop by hop, many take one each or part of a wavefront; fanouts of every group
    # width; a frontier of more than 65,536 rows streams its long rows instead of making them tile by tile; with the first hop from
    # tables and, by default, from the weights
    from helpers import graph_from_degrees
    from skywalker_amd import capi
    rng = np.random.default_rng(78)
    degs = [0, 1, 2, 3, 4, 5, 16, 17, 32, 33, 34, 63, 64, 65, 66, 200, 600, 1500, 3000, 5200, 8190, 9001, 25003, 66001, 530001]
    degs += list(rng.integers(0, 90, 400)) + ([1, 2, 3] * 24000 if n > 65536 else [])
    xadj, adjncy, w = graph_from_degrees(degs, rng, "sparse")
    V = len(xadj) - 1
    seeds = (np.append(V, rng.permutation(V)) if n > 65536 else rng.integers(0, V + 1, n)).astype(np.uint32)[:n]
    if n > 65536:
        seeds[1:26] = np.arange(25)
    lps, slen = capi.sample_layout(fanout)
    g = capi.Graph.upload(xadj, adjncy, w)
    g.set_option("stream_min_edges", 0)
    g.set_option("sample_distinct", int(distinct))
    g.set_option("online_direct", 0)
    tabled = g.sample_online(seeds, fanout, 37)
    g.set_option("online_direct", -1)
    on = g.sample_online(seeds, fanout, 37)
    g.build_tables()
    off = g.sample_offline(seeds, fanout, 37)
    prob, alias, _ = g.tables()
    want = orc.sample_offline(xadj, adjncy, prob, alias, seeds, fanout, 37, distinct=distinct)
    for data, sl, sampled, _ in (tabled, on, off):
        assert np.array_equal(sl.to_host((n, slen)), want[1]) and np.array_equal(data.to_host((n, lps)), want[0])
        assert sampled == want[2]
    g.free()


def test_other_calls_between_the_steps_of_a_session(orc):
    # a larger batch with more hops, and a second session, on the same graph between the steps: buffers of the first
    # session neither move nor change (what the lists and counts hold: the next test)
    import ctypes as C
    from helpers import graph_from_degrees
    from skywalker_amd import capi
    rng = np.random.default_rng(79)
    degs = list(rng.integers(0, 60, 3000)) + [300, 700, 3000, 6000, 9000, 70001] * 3
    rng.shuffle(degs)
    xadj, adjncy, w = graph_from_degrees(degs, rng, "lognormal")
    V = len(xadj) - 1
    g = capi.Graph.upload(xadj, adjncy, w)
    L, fan = capi.lib(), np.array([1, 5, 4, 2], np.uint32)
    lps, slen = capi.sample_layout(fan)
    sessions = []
    for n in (40, 900):
        seeds = rng.integers(0, V, n).astype(np.uint32)
        seeds_d = capi.DeviceArray.from_host(seeds)
        data, sl = capi.DeviceArray(n * lps, np.uint32, fill=0xFFFFFFFF), capi.DeviceArray(n * slen, np.uint32, fill=0)
        sess = C.c_void_p()
        assert L.sky_sample_session_begin(g.h, seeds_d.ptr, C.c_uint32(n), fan.ctypes.data_as(C.c_void_p), C.c_uint32(len(fan)),
                                          C.c_uint64(41), data.ptr, sl.ptr, C.byref(sess)) == 0
        sessions.append((n, seeds, seeds_d, data, sl, sess))
    big = rng.integers(0, V, 20000).astype(np.uint32)
    for hop in range(3):
        for _, _, _, _, _, sess in sessions:
            lst, cnt, upper = C.c_void_p(), C.c_void_p(), C.c_uint32()
            assert L.sky_sample_session_frontier(sess, C.c_uint32(hop), C.byref(lst), C.byref(cnt), C.byref(upper)) == 0
        got = g.sample_online(big[:20000 >> (2 * (2 - hop))], [1, 3, 2, 2, 2], 43)
        want = orc.sample_online(xadj, adjncy, w, big[:20000 >> (2 * (2 - hop))], [1, 3, 2, 2, 2], 43)
        assert np.array_equal(got[0].to_host(want[0].shape), want[0]) and got[2] == want[2]
        for _, _, _, _, _, sess in sessions:
            assert L.sky_sample_session_hop(sess, C.c_uint32(hop), None) == 0
    for n, seeds, _, data, sl, sess in sessions:
        sampled, sec = C.c_uint64(), C.c_double()
        assert L.sky_sample_session_end(sess, C.byref(sampled), C.byref(sec)) == 0
        want = orc.sample_online(xadj, adjncy, w, seeds, fan, 41)
        assert np.array_equal(data.to_host((n, lps)), want[0]) and np.array_equal(sl.to_host((n, slen)), want[1])
        assert sampled.value == want[2]
    g.free()


def open_session(capi, g, seeds, fan, seed, sl_fill=0):
    """begin: (session, seeds, fanouts, data, sample_lengths), everything that has to stay alive."""
    import ctypes as C
    lps, slen = capi.sample_layout(fan)
    seeds_d, fan = capi.DeviceArray.from_host(seeds), np.array(fan, np.uint32)
    data = capi.DeviceArray(len(seeds) * lps, np.uint32, fill=capi.FILL)
    sl = capi.DeviceArray(len(seeds) * slen, np.uint32, fill=sl_fill)
    sess = C.c_void_p()
    capi._ck(capi.lib().sky_sample_session_begin(g.h, seeds_d.ptr, C.c_uint32(len(seeds)), capi._p(fan), C.c_uint32(len(fan)),
                                                 C.c_uint64(seed), data.ptr, sl.ptr, C.byref(sess)))
    return sess, seeds_d, fan, data, sl


def session_frontier(capi, sess, hop):
    """Device addresses of list and count, and the bound."""
    import ctypes as C
    lst, cnt, upper = C.c_void_p(), C.c_void_p(), C.c_uint32()
    capi._ck(capi.lib().sky_sample_session_frontier(sess, C.c_uint32(hop), C.byref(lst), C.byref(cnt), C.byref(upper)))
    return lst, cnt, upper.value


def session_end(capi, sess):
    import ctypes as C
    sampled, sec = C.c_uint64(), C.c_double()
    capi._ck(capi.lib().sky_sample_session_end(sess, C.byref(sampled), C.byref(sec)))
    return sampled.value, sec.value


def read_list(capi, lst, cnt, room):
    n = np.empty(1, np.uint32)
    capi._ck(capi.lib().sky_memcpy_d2h(capi._p(n), cnt, 4))
    assert n[0] <= room
    out = np.empty(int(n[0]), np.uint32)
    capi._ck(capi.lib().sky_memcpy_d2h(capi._p(out), lst, int(out.nbytes)))
    return out


def parents_by_hop(data, fan, V):
    """Distinct vertices of every hop that no hop before held, from the sampled blocks."""
    seen, out, off, width = np.zeros(0, np.uint32), [], 0, 1
    for h in range(len(fan) - 1):
        width *= int(fan[h])
        block = np.unique(data[:, off:off + width])
        fresh = np.setdiff1d(block[block < V], seen)
        out.append(fresh)
        seen = np.union1d(seen, fresh)
        off += width
    return out


@pytest.mark.parametrize("device_sized", [1, 0])
def test_lists_and_counts_of_sessions_open_at_the_same_time(orc, device_sized):
    # two sessions at the same hop, other calls before the lists are read: every list holds the distinct parents of its own
    # session, and weights given for the listed rows alone are all that the builds need
    import ctypes as C
    from skywalker_amd import capi
    rng = np.random.default_rng(80)
    degs = list(rng.integers(0, 60, 3000)) + [300, 700, 3000, 6000, 9000, 70001] * 3
    rng.shuffle(degs)
    xadj, adjncy, w = graph_from_degrees(degs, rng, "lognormal")
    V, fan = len(xadj) - 1, [1, 5, 4, 2]
    lps, slen = capi.sample_layout(fan)
    g = capi.Graph.upload(xadj, adjncy, w)
    g.set_option("online_device_sized", device_sized)
    g.set_option("online_full_build", 0)
    some = rng.integers(0, V, 700).astype(np.uint32)
    runs = []
    for n in (40, V):  # the second session's first frontier is every vertex: its list is full
        seeds = rng.integers(0, V, n).astype(np.uint32) if n < V else np.arange(V, dtype=np.uint32)
        want = orc.sample_online(xadj, adjncy, w, seeds, fan, 41)
        runs.append((seeds, want, parents_by_hop(want[0], fan, V), np.zeros_like(w), open_session(capi, g, seeds, fan, 41)))
    for hop in range(3):
        lists = [session_frontier(capi, s[0], hop) for _, _, _, _, s in runs]
        g.walk_online(capi.BIAS_STATIC, 1.0, 1.0, some, 4, 0.0, 5)
        got = g.sample_online(some, [1, 3, 2], 43)
        want = orc.sample_online(xadj, adjncy, w, some, [1, 3, 2], 43)
        assert np.array_equal(got[0].to_host(want[0].shape), want[0]) and got[2] == want[2]
        for (seeds, _, parents, mine, s), (lst, cnt, upper) in zip(runs, lists):
            listed = read_list(capi, lst, cnt, upper)
            assert np.array_equal(np.sort(listed), parents[hop])
            for v in listed:
                mine[xadj[v]:xadj[v + 1]] = w[xadj[v]:xadj[v + 1]]
            w_d = capi.DeviceArray.from_host(mine)
            capi._ck(capi.lib().sky_sample_session_hop(s[0], C.c_uint32(hop), w_d.ptr))
    for seeds, want, _, _, s in runs:
        sampled, sec = session_end(capi, s[0])
        n = len(seeds)
        assert np.array_equal(s[3].to_host((n, lps)), want[0]) and np.array_equal(s[4].to_host((n, slen)), want[1])
        assert sampled == want[2] and 0 < sec < 60
    g.free()


@pytest.mark.parametrize("n,fan", [(40, [1, 5, 4]), (3, [1, 64, 64])])
@pytest.mark.parametrize("distinct", [0, 1])
def test_session_ended_before_its_last_hop(orc, n, fan, distinct):
    # the count and the lengths are those of the hops that were drawn, whatever the caller's array held before; totals added
    # up by the workgroups of the start vertices (40) and by the lengths (3 x 64 x 64, several workgroups each)
    import ctypes as C
    from skywalker_amd import capi
    rng = np.random.default_rng(81)
    xadj, adjncy, w = graph_from_degrees(rng.integers(3, 90, 500), rng, "lognormal")
    seeds = rng.integers(0, 500, n).astype(np.uint32)
    prob, alias, _ = orc.alias_build(xadj, w)
    whole = orc.sample_offline(xadj, adjncy, prob, alias, seeds, fan, 47, distinct=bool(distinct))
    g = capi.Graph.upload(xadj, adjncy, w)
    g.set_option("sample_distinct", distinct)
    for drawn in (0, 1):
        s = open_session(capi, g, seeds, fan, 47, sl_fill=7)
        for hop in range(drawn):
            session_frontier(capi, s[0], hop)
            capi._ck(capi.lib().sky_sample_session_hop(s[0], C.c_uint32(hop), None))
        sampled, _ = session_end(capi, s[0])
        sl = whole[1].copy()
        sl[:, drawn:] = 0  # one length per start vertex at hop 0
        assert np.array_equal(s[4].to_host(sl.shape), sl) and sampled == int(sl.sum())
    g.free()


def test_online_calls_on_a_graph_without_vertices_and_without_tables(orc):
    from skywalker_amd import capi
    none = np.zeros(0, np.uint32)
    for V in (0, 300):
        g = capi.Graph.upload(np.zeros(V + 1, np.uint32), none, np.zeros(0, np.float32))
        for device_sized in (1, 0):
            g.set_option("online_device_sized", device_sized)
            assert g.sample_online(none, [1, 3, 2], 1)[2] == 0
            assert g.sample_session(none, [1, 3, 2], 1)[2] == 0
        assert g.walk_online(capi.BIAS_STATIC, 1.0, 1.0, none, 4, 0.0, 1)[2] == 0
        assert g.walk_online(capi.BIAS_NODE2VEC, 2.0, 0.5, none, 4, 0.0, 1)[2] == 0
        g.free()


def test_knobs_changed_between_the_steps_of_a_session(orc):
    # stream_min_edges decides which rows a build makes tile by tile; a session goes on as it began when the knob changes and
    # another call lays the graph's rows out anew
    import ctypes as C
    from skywalker_amd import capi
    rng = np.random.default_rng(82)
    degs = list(rng.integers(0, 60, 2000)) + [300, 3000, 6000, 9000, 25000, 70001] * 3
    rng.shuffle(degs)
    xadj, adjncy, w = graph_from_degrees(degs, rng, "lognormal")
    V, fan = len(xadj) - 1, [1, 5, 4, 2]
    lps, slen = capi.sample_layout(fan)
    g = capi.Graph.upload(xadj, adjncy, w)
    g.set_option("online_full_build", 0)
    seeds = np.arange(V, dtype=np.uint32)
    want = orc.sample_online(xadj, adjncy, w, seeds, fan, 53)
    some = rng.integers(0, V, 300).astype(np.uint32)

    def elsewhere(value):
        g.set_option("stream_min_edges", value)
        got, expect = g.walk_online(capi.BIAS_STATIC, 1.0, 1.0, some, 6, 0.0, 5), orc.walk_online(xadj, adjncy, w, 0, 1.0, 1.0, some, 6, 0.0, 5)
        assert np.array_equal(got[0].to_host(expect[0].shape), expect[0])
    s = open_session(capi, g, seeds, fan, 53)
    for hop in range(3):
        elsewhere(0 if hop % 2 else 1 << 30)
        session_frontier(capi, s[0], hop)
        elsewhere(1 << 30 if hop % 2 else 0)
        capi._ck(capi.lib().sky_sample_session_hop(s[0], C.c_uint32(hop), None))
    sampled, _ = session_end(capi, s[0])
    assert np.array_equal(s[3].to_host((V, lps)), want[0]) and np.array_equal(s[4].to_host((V, slen)), want[1])
    assert sampled == want[2]
    g.free()


def test_rows_that_other_calls_build_between_the_hops_of_a_session(orc):
    # weights are given for the rows that a hop lists and no others, as the interface asks: a long row that hop 0 has built,
    # and that another call builds as well before hop 1 draws from it again, must not be built from hop 1's weights
    import ctypes as C
    from skywalker_amd import capi
    rng = np.random.default_rng(83)
    degs = list(rng.integers(3, 60, 400)) + [9000, 30000, 70001, 600001]
    xadj, adjncy, w = graph_from_degrees(degs, rng, "lognormal")
    V, fan = len(xadj) - 1, [1, 8, 4]
    adjncy[xadj[:-1]] = V - 4 + np.arange(V) % 4  # every row leads to a long one ...
    w[xadj[:-1]] = 1000.0                                            # ... and mostly there
    lps, slen = capi.sample_layout(fan)
    seeds = np.arange(V - 60, V, dtype=np.uint32)
    want = orc.sample_online(xadj, adjncy, w, seeds, fan, 59)
    assert np.isin(want[0][:, 1:9], np.arange(V - 4, V)).any()
    g = capi.Graph.upload(xadj, adjncy, w)
    s = open_session(capi, g, seeds, fan, 59)
    for hop in range(2):
        lst, cnt, upper = session_frontier(capi, s[0], hop)
        mine = np.zeros_like(w)
        for v in read_list(capi, lst, cnt, upper):
            mine[xadj[v]:xadj[v + 1]] = w[xadj[v]:xadj[v + 1]]
        w_d = capi.DeviceArray.from_host(mine)
        if hop:
            g.sample_online(seeds, [1, 2], 61)
        capi._ck(capi.lib().sky_sample_session_hop(s[0], C.c_uint32(hop), w_d.ptr))
    sampled, _ = session_end(capi, s[0])
    assert np.array_equal(s[3].to_host((60, lps)), want[0]) and np.array_equal(s[4].to_host((60, slen)), want[1])
    assert sampled == want[2]
    g.free()


def test_row_lists_made_anew_leave_the_flags_of_a_session_alone(orc):
    # a row without weight that a session has built stays without children when another call makes the graph's row lists anew
    import ctypes as C
    from skywalker_amd import capi
    rng = np.random.default_rng(84)
    degs, fan = [40] * 8 + [1] * 8, [1, 64, 64]  # fanouts above the degree: all neighbours of a row with weight
    xadj, adjncy, w = graph_from_degrees(degs, rng, "uniform")
    w[:8 * 40] = 0.0
    adjncy[8 * 40:] = np.arange(8)  # hop 0 leads from the rows of one entry to those without weight
    lps, slen = capi.sample_layout(fan)
    seeds = np.arange(16, dtype=np.uint32)
    want = orc.sample_online(xadj, adjncy, w, seeds, fan, 67)
    g = capi.Graph.upload(xadj, adjncy, w)
    g.set_option("online_full_build", 0)
    s = open_session(capi, g, seeds, fan, 67)
    for hop in range(2):
        session_frontier(capi, s[0], hop)
        capi._ck(capi.lib().sky_sample_session_hop(s[0], C.c_uint32(hop), None))
        g.set_option("stream_min_edges", 7 + hop)
        g.walk_online(capi.BIAS_STATIC, 1.0, 1.0, seeds[15:], 1, 0.0, 5)
    sampled, _ = session_end(capi, s[0])
    assert np.array_equal(s[4].to_host((16, slen)), want[1]) and np.array_equal(s[3].to_host((16, lps)), want[0])
    assert sampled == want[2] == 8
    g.free()


def test_hop_of_a_session_taken_once_more(orc):
    # a frontier of more than 65,536 rows, 1,100 of which are streamed by the workgroup that is first free: the second time, from other
    # weights, every one of them is built again
    import ctypes as C
    from skywalker_amd import capi
    rng = np.random.default_rng(85)
    degs = list(rng.integers(8190, 9500, 1100)) + list(rng.integers(1, 4, 70000))
    rng.shuffle(degs)
    xadj = np.concatenate([[0], np.cumsum(degs)]).astype(np.uint32)
    V, E, fan = len(degs), int(xadj[-1]), [1, 3]
    adjncy = rng.integers(0, V, E, dtype=np.uint32)
    w = [weights(E, rng, "lognormal2") for _ in range(2)]
    seeds = rng.permutation(V).astype(np.uint32)
    lps, slen = capi.sample_layout(fan)
    g = capi.Graph.upload(xadj, adjncy, w[0])
    s = open_session(capi, g, seeds, fan, 71)
    session_frontier(capi, s[0], 0)
    for x in w:
        w_d = capi.DeviceArray.from_host(x)
        capi._ck(capi.lib().sky_sample_session_hop(s[0], C.c_uint32(0), w_d.ptr))
        capi.synchronize()
    session_end(capi, s[0])
    want = orc.sample_online(xadj, adjncy, w[1], seeds, fan, 71)
    assert np.array_equal(s[4].to_host((V, slen)), want[1]) and np.array_equal(s[3].to_host((V, lps)), want[0])
    g.free()


@pytest.mark.parametrize("fanout", [[1, 20], [1, 5, 3], [1, 70], [1, 600], [1, 1]])
@pytest.mark.parametrize("dist,seeds_n", [("lognormal2", 333), ("sparse", 1601), ("nearequal", 40)])
def test_children_drawn_from_the_weights(orc, fanout, dist, seeds_n):
    # without tables, a wavefront or a workgroup a slot: rows around the fan-out, around 4 and 16 slots a thread and around the rows that a
    # workgroup shares; rows without weight, and with surpluses beyond 64 bits; workgroups partly empty; start vertices that do not exist
    from skywalker_amd import capi
    rng = np.random.default_rng(53)
    degs = [0, 1, 2, 3, 4, 5, 19, 20, 21, 63, 64, 65, 69, 70, 71, 255, 256, 257, 260, 511, 513, 599, 600, 601, 1021, 1023, 1024, 1025,
            2047, 2048, 2049, 4097, 8191, 8193, 40001] + list(rng.integers(1, 700, 40))
    xadj, adjncy, w = graph_from_degrees(degs, rng, dist)
    n = len(degs)
    for v in range(0, n, 3):
        if dist == "sparse":
            w[xadj[v]:xadj[v + 1]] *= np.float32(1e-19)
    for v in (7, 20, 31):
        w[xadj[v]:xadj[v + 1]] = 0.0
    seeds = np.append((np.arange(seeds_n - 1) * 7) % n, n + 5).astype(np.uint32)
    lps, slen = capi.sample_layout(fanout)
    want = orc.sample_online(xadj, adjncy, w, seeds, fanout, 61)
    g = capi.Graph.upload(xadj, adjncy, w)
    for mode in (1, -1, 0):  # whatever the rows, unless they are long, never
        g.set_option("online_direct", mode)
        d, sl, sampled, _ = g.sample_online(seeds, fanout, 61)
        assert np.array_equal(sl.to_host((seeds_n, slen)), want[1]) and np.array_equal(d.to_host((seeds_n, lps)), want[0])
        assert sampled == want[2]
    g.free()


@pytest.mark.parametrize("fanout", [[1, 20], [1, 10, 10], [1, 10, 300]])
@pytest.mark.parametrize("longest", [40001, 60001])
def test_parents_whose_rows_are_too_long_to_draw_from_the_weights(orc, fanout, longest):
    # one long row again and again, beside others, and behind rows of one entry: the first hop is drawn from tables after all, or the
    # second where the longest row is short enough for a call that begins without any
    from skywalker_amd import capi
    rng = np.random.default_rng(89)
    degs = np.full(105001, 10)
    degs[0], degs[1:5001] = longest, 1
    xadj = np.concatenate([[0], np.cumsum(degs)]).astype(np.uint32)
    V, E = len(degs), int(xadj[-1])
    adjncy = rng.integers(0, V, E, dtype=np.uint32)
    adjncy[longest:longest + 5000] = 0  # rows 1 to 5000 lead to the long one
    w = weights(E, rng, "lognormal2")
    lps, slen = capi.sample_layout(fanout)
    g = capi.Graph.upload(xadj, adjncy, w)
    short = rng.integers(5001, V, 4000).astype(np.uint32)
    mixed = short.copy()
    mixed[3000] = 0
    for seeds in (np.zeros(30, np.uint32), np.zeros(3000, np.uint32), np.arange(1, 31, dtype=np.uint32), short[:30], short, mixed):
        want = orc.sample_online(xadj, adjncy, w, seeds, fanout, 73)
        for _ in range(2):
            d, sl, sampled, _ = g.sample_online(seeds, fanout, 73)
            assert np.array_equal(sl.to_host((len(seeds), slen)), want[1]) and np.array_equal(d.to_host((len(seeds), lps)), want[0])
            assert sampled == want[2]
    g.free()


def test_a_vertex_that_starts_every_sample_is_not_swept_for_each_of_them():
    # 8,192 times a row of 60,000 entries: its table takes microseconds, and by default it is made once
    from skywalker_amd import capi
    rng = np.random.default_rng(90)
    degs = np.full(100001, 10)
    degs[0] = 60000
    xadj = np.concatenate([[0], np.cumsum(degs)]).astype(np.uint32)
    E = int(xadj[-1])
    g = capi.Graph.upload(xadj, rng.integers(0, len(degs), E, dtype=np.uint32), weights(E, rng, "lognormal"))
    seeds = np.zeros(8192, np.uint32)

    def seconds(mode):
        g.set_option("online_direct", mode)
        return min(g.sample_online(seeds, [1, 20], 1)[3] for _ in range(5))
    never, default, always = seconds(0), seconds(-1), seconds(1)
    print("never %.1f us, by default %.1f us, always %.1f us" % (never * 1e6, default * 1e6, always * 1e6))
    assert default < 2 * never and 2 * default < always
    g.free()


@pytest.mark.parametrize("asked", ["one", "tenth", "all", "none"])
def test_frontiers_that_ask_for_some_of_many_rows_made_by_tiles(orc, asked):
    # 500 rows of 9 to 13 tiles each, of which the frontier wants some; fewer than the 8,192 tiles from which the rows go out beside the passes
    from skywalker_amd import capi
    rng = np.random.default_rng(91)
    degs = np.concatenate([rng.integers(8190, 12500, 500), np.full(20000, 3)])
    rng.shuffle(degs)
    xadj, adjncy, w = graph_from_degrees(degs, rng, "lognormal2")
    long_rows = np.flatnonzero(degs > 3).astype(np.uint32)
    long_rows = {"one": long_rows[250:251], "tenth": long_rows[::10], "all": long_rows, "none": long_rows[:0]}[asked]
    seeds = np.concatenate([long_rows, rng.permutation(np.flatnonzero(degs == 3))[:2000].astype(np.uint32)])
    fan = [1, 7]
    lps, slen = capi.sample_layout(fan)
    want = orc.sample_online(xadj, adjncy, w, seeds, fan, 75)
    g = capi.Graph.upload(xadj, adjncy, w)
    g.set_option("online_direct", 0)
    for _ in range(2):
        d, sl, sampled, _ = g.sample_online(seeds, fan, 75)
        assert np.array_equal(sl.to_host((len(seeds), slen)), want[1]) and np.array_equal(d.to_host((len(seeds), lps)), want[0])
        assert sampled == want[2]
    g.free()


@pytest.mark.parametrize("kind", ["one", "two", "pairs", "far"])
def test_vertices_that_a_workgroup_of_the_collection_meets_again(orc, kind):
    # every lane the same vertex, two of them in turn, every vertex twice in a row, and vertices that share their places in LDS (the
    # bits of 4,096 places apart, by the factor's inverse)
    from skywalker_amd import capi
    rng = np.random.default_rng(92)
    V, n = 1 << 15, 2500
    xadj, adjncy, w = graph_from_degrees(rng.integers(1, 9, V), rng, "uniform")
    inverse = pow(2654435769, -1, V)
    seeds = {"one": np.full(n, 77), "two": np.arange(n) % 2, "pairs": np.arange(n) // 2,
             "far": np.array([(5 + 4096 * (i % 8)) * inverse % V for i in range(n)])}[kind].astype(np.uint32)
    fan = [1, 2]
    lps, slen = capi.sample_layout(fan)
    want = orc.sample_online(xadj, adjncy, w, seeds, fan, 76)
    for mode in (1, 0):  # by class in device-sized builds, and as a list
        g = capi.Graph.upload(xadj, adjncy, w)
        g.set_option("online_direct", 0)
        g.set_option("online_device_sized", mode)
        d, sl, sampled, _ = g.sample_online(seeds, fan, 76)
        assert np.array_equal(sl.to_host((n, slen)), want[1]) and np.array_equal(d.to_host((n, lps)), want[0]) and sampled == want[2]
        g.free()


@pytest.fixture(scope="module")
def many_tiles():
    # 1,200 rows of 9 to 13 tiles each: 14,500 tiles, more than a launch of one workgroup a row holds rows at a time, and enough for launches of
    # their own beside the rows of a frontier
    rng = np.random.default_rng(93)
    degs = np.concatenate([rng.integers(8190, 12500, 1200), rng.integers(33, 5000, 300), np.full(20000, 3)])
    rng.shuffle(degs)
    xadj, adjncy, w = graph_from_degrees(degs, rng, "lognormal2")
    long_rows = np.flatnonzero(degs >= 8190).astype(np.uint32)
    adjncy[rng.random(len(adjncy)) < 0.5] = rng.choice(long_rows, 1)[0]  # a row that is met at the next hop too
    return xadj, adjncy, w, long_rows, np.flatnonzero(degs < 8190).astype(np.uint32)


@pytest.mark.parametrize("streams", [1, 0])
@pytest.mark.parametrize("asked", ["one", "tenth", "all", "none"])
def test_frontiers_beside_the_passes_over_many_tiles(orc, many_tiles, asked, streams):
    # two hops, so that a build follows the build before on the same words; the third call finds what the first two left
    from skywalker_amd import capi
    xadj, adjncy, w, long_rows, others = many_tiles
    rng = np.random.default_rng(94)
    mine = {"one": long_rows[600:601], "tenth": long_rows[::10], "all": long_rows, "none": long_rows[:0]}[asked]
    seeds = np.concatenate([mine, rng.permutation(others)[:2000].astype(np.uint32)])
    fan = [1, 7, 3]
    lps, slen = capi.sample_layout(fan)
    want = orc.sample_online(xadj, adjncy, w, seeds, fan, 77)
    g = capi.Graph.upload(xadj, adjncy, w)
    g.set_option("online_direct", 0)
    g.set_option("build_streams", streams)
    for _ in range(3):
        d, sl, sampled, _ = g.sample_online(seeds, fan, 77)
        assert np.array_equal(sl.to_host((len(seeds), slen)), want[1]) and np.array_equal(d.to_host((len(seeds), lps)), want[0])
        assert sampled == want[2]
    g.free()


@pytest.mark.parametrize("streams", [1, 0])
def test_sessions_beside_the_passes_over_many_tiles(orc, many_tiles, streams):
    # weights of the caller's, other ones in the graph; every hop built and drawn twice, the second time from the weights that count
    import ctypes as C
    from skywalker_amd import capi
    xadj, adjncy, w, long_rows, others = many_tiles
    seeds = np.concatenate([long_rows[::3], others[:500]])
    fan = [1, 5, 2]
    lps, slen = capi.sample_layout(fan)
    want = orc.sample_online(xadj, adjncy, w, seeds, fan, 78)
    g = capi.Graph.upload(xadj, adjncy, w[::-1].copy())
    g.set_option("build_streams", streams)
    wrong, right = capi.DeviceArray.from_host(np.roll(w, 7)), capi.DeviceArray.from_host(w)
    for _ in range(2):
        s = open_session(capi, g, seeds, fan, 78)
        for hop in range(2):
            session_frontier(capi, s[0], hop)
            for weights_d in (wrong, right):
                capi._ck(capi.lib().sky_sample_session_hop(s[0], C.c_uint32(hop), weights_d.ptr))
        session_end(capi, s[0])
        assert np.array_equal(s[4].to_host((len(seeds), slen)), want[1]) and np.array_equal(s[3].to_host((len(seeds), lps)), want[0])
    g.free()
