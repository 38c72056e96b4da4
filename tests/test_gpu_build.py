"""Offline alias build on the GPU (through the C-ABI) against the CPU oracle: bit-exact tables,
and the reconstruction invariant on every row."""
import numpy as np
import pytest

from helpers import graph_from_degrees

pytestmark = pytest.mark.gpu
TOL = 1e-6

# degrees that straddle every dispatch class boundary of the build
EDGE_DEGREES = [0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 16, 17, 22, 23, 24, 25, 28, 29, 30, 32, 33, 46, 47, 48,
                49, 60, 61, 62, 63, 64, 65, 66, 67, 68, 94, 95, 96, 97, 124, 125, 126, 127, 190, 191, 192, 193, 253, 254, 255, 256, 257, 380, 381, 382, 383, 509, 510, 511, 764, 765, 766, 767, 1021,
                1022, 1023, 1024, 1025, 4093, 4094, 4095, 4096, 4097, 5116, 5117, 5118, 5119, 5120, 5121, 8189, 8190, 8191, 8192, 8193, 16380, 16381, 16382, 16383, 20000, 70001, 128, 129, 130, 144, 145, 159, 160, 161, 162, 34, 35, 36, 45]


def build_and_compare(orc, xadj, adjncy, w, label):
    from skywalker_amd import capi
    print("case", label, "V", len(xadj) - 1, "E", len(w), flush=True)
    oprob, oalias, ovalid = orc.alias_build(xadj, w)
    deg = np.diff(xadj)
    # rows of 8190..524287 entries: once through their own kernel, once (the default for so few of them)
    # through the tile-parallel path
    routes = (0, 4000000) if ((deg >= 8190) & (deg <= 524287)).any() else (4000000,)
    # rows of at most 32 entries: by degree class (the default below 2^25 rows), and by the kernel that walks the
    # vertices in order
    for stream_min_edges, small_in_place in [(r, 0) for r in routes] + [(routes[0], 1)]:
        g = capi.Graph.upload(xadj, adjncy, w)
        # knobs of this graph alone: nothing to restore, whatever happens below
        g.set_option("stream_min_edges", stream_min_edges)
        g.set_option("stream_wide_min_edges", stream_min_edges)  # 0: also the rows above 65533 entries are streamed
        g.set_option("small_in_place", small_in_place)
        g.build_tables()
        prob, alias, valid = g.tables()
        g.free()
        st = orc.alias_check(xadj, w, prob, alias, valid)
        assert st["bad_valid"] == 0 and st["bad_range"] == 0 and st["bad_invalid"] == 0, st
        assert st["max_rel_err"] < TOL, st
        bad = np.flatnonzero((prob != oprob) | (alias != oalias))
        if len(bad):
            v = int(np.searchsorted(xadj, bad[0], side="right") - 1)
            raise AssertionError("%s (stream_min_edges %d, small_in_place %d): %d entries differ from the oracle, first "
                                 "at slot %d (vertex %d, degree %d)" % (label, stream_min_edges, small_in_place, len(bad),
                                                                        bad[0], v, xadj[v + 1] - xadj[v]))
        assert np.array_equal(valid, ovalid)


@pytest.mark.parametrize("dist", ["lognormal", "uniform", "unit", "lognormal2", "equal", "nearequal", "sparse"])
def test_every_degree_class(orc, dist):
    rng = np.random.default_rng(11)
    degs = EDGE_DEGREES + list(rng.integers(1, 300, 400)) + list(rng.integers(300, 6000, 30))
    rng.shuffle(degs)
    xadj, adjncy, w = graph_from_degrees(degs, rng, dist, V=len(degs) + 7)
    build_and_compare(orc, xadj, adjncy, w, "classes/" + dist)


def test_class_kernels_over_side_streams_give_the_same_table(orc):
    # a build of 2 M .. 1 G entries spreads its class kernels over side streams; option build_streams = 0 keeps
    # them on the graph's stream
    from skywalker_amd import capi
    rng = np.random.default_rng(21)
    degs = EDGE_DEGREES[:60] + list(rng.integers(1, 300, 3000)) + list(rng.integers(300, 9000, 400)) + [30_000, 70_000, 600_000]
    rng.shuffle(degs)
    xadj, adjncy, w = graph_from_degrees(degs, rng, "lognormal")
    assert 2_000_000 <= len(w) < (1 << 30)
    for on in (0, 1):
        capi.set_option("build_streams", on)
        try:
            for rep in range(2):  # twice: the second build finds the side streams and their events in place
                build_and_compare(orc, xadj, adjncy, w, "side streams %d" % on)
        finally:
            capi.set_option("build_streams", 1)


def test_unaligned_row_starts(orc):
    # rows of every residue mod 4 in front of each LDS-class row
    rng = np.random.default_rng(5)
    degs = []
    for d in (70, 254, 700, 1021, 3000, 4093, 5117, 5118, 8000, 8189, 9000):
        for pad in (1, 2, 3, 5):
            degs += [pad, d]
    xadj, adjncy, w = graph_from_degrees(degs, rng, "lognormal")
    build_and_compare(orc, xadj, adjncy, w, "unaligned")


def test_all_zero_and_empty_rows(orc):
    rng = np.random.default_rng(2)
    degs = [0, 5, 0, 40, 100, 1, 2, 3000, 9000, 0]
    xadj, adjncy, w = graph_from_degrees(degs, rng, "uniform")
    for v in (1, 3, 4, 5, 6, 7, 8):
        if v % 2 == 1 or v == 8:
            w[xadj[v]:xadj[v + 1]] = 0.0
    build_and_compare(orc, xadj, adjncy, w, "zero rows")


def test_hub_row(orc):
    rng = np.random.default_rng(3)
    xadj, adjncy, w = graph_from_degrees([1_200_000, 3, 90_000], rng, "lognormal2", V=4096)
    build_and_compare(orc, xadj, adjncy, w, "hub")


def test_config1_rmat_s16(orc):
    xadj, adjncy = orc.rmat_csr(16, 16, 42)
    w = orc.gen_weights(orc.W_UNIFORM, 42, len(adjncy), 1.0, 100.0)
    build_and_compare(orc, xadj, adjncy, w, "config1")


def test_rebuild_is_idempotent(orc):
    from skywalker_amd import capi
    xadj, adjncy = orc.rmat_csr(12, 8, 9)
    w = orc.gen_weights(orc.W_UNIT, 9, len(adjncy))
    g = capi.Graph.upload(xadj, adjncy, w)
    g.build_tables()
    a = g.tables()
    g.build_tables()
    b = g.tables()
    g.free()
    for x, y in zip(a, b):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("exact", [True, False])
def test_build_from_a_callers_weight_array(orc, exact):
    # sky_alias_build_from_weights with weights other than the graph's own: in device memory that ends with the
    # last of its E floats (E a multiple of 1024, ending in a short row whose 16-byte loads reach past the last
    # weight: the library copies such an array into a padded one), and in an array from sky_device_malloc, which
    # adds 16 bytes to every allocation (read where it lies)
    from skywalker_amd import capi
    import ctypes
    rng = np.random.default_rng(41)
    degs = list(rng.integers(1, 200, 300)) + [3000, 9000, 70, 33, 17]
    fill = (-sum(degs) - 5) % 1024
    degs += [fill, 5]
    xadj, adjncy, w = graph_from_degrees(degs, rng, "uniform")
    E = len(w)
    assert E % 1024 == 0 and xadj[-1] == E and xadj[len(degs)] - xadj[len(degs) - 1] == 5
    other = rng.lognormal(0, 2, E).astype(np.float32)
    g = capi.Graph.upload(xadj, adjncy, w)
    # the allocation holds 4 * (E + 8) + 16 bytes: 32 bytes in, exactly E floats are left
    dev = capi.DeviceArray(E + 8 if exact else E, np.float32)

    class View:
        ptr = ctypes.c_void_p(dev.ptr.value + 32) if exact else dev.ptr
    capi._ck(capi.lib().sky_memcpy_h2d(View.ptr, capi._p(other), E * 4))
    for rep in range(2):  # the second call finds the padded copy in place
        g.build_tables_from_weights(View)
        prob, alias, valid = g.tables()
        oprob, oalias, ovalid = orc.alias_build(xadj, other)
        assert np.array_equal(prob, oprob) and np.array_equal(alias, oalias) and np.array_equal(valid, ovalid)
    assert np.array_equal(g.download()[2], w)  # the graph's own weights are left as they are
    g.build_tables()
    prob, alias, valid = g.tables()
    oprob, oalias, ovalid = orc.alias_build(xadj, w)
    assert np.array_equal(prob, oprob) and np.array_equal(alias, oalias) and np.array_equal(valid, ovalid)
    dev.free()
    g.free()


def test_bad_arguments_are_reported(orc):
    from skywalker_amd import capi
    xadj = np.array([0, 2, 1], np.uint32)  # not monotone
    with pytest.raises(capi.SkyError):
        capi.Graph.upload(xadj, np.zeros(1, np.uint32), np.ones(1, np.float32))
    xadj = np.array([0, 1], np.uint32)
    with pytest.raises(capi.SkyError):
        capi.Graph.upload(xadj, np.array([5], np.uint32), np.ones(1, np.float32))  # neighbour out of range
    g = capi.Graph.upload(np.array([0, 1, 1], np.uint32), np.array([1], np.uint32), np.ones(1, np.float32))
    with pytest.raises(capi.SkyError):
        g.walk_offline(np.array([0], np.uint32), 4, 0.0, 1)  # tables not built
    g.free()


@pytest.mark.parametrize("dist", ["lognormal2", "nearequal", "sparse", "fewlights", "fewheavies"])
def test_rows_built_tile_by_tile(orc, dist):
    # rows beyond one workgroup's LDS: 8 to 320 tiles, starts of every alignment
    from helpers import weights
    rng = np.random.default_rng(21)
    degs = [4094, 4097, 7, 5121, 8190, 1, 8193, 2, 12288, 3, 12289, 40000, 5, 100001, 330000]
    xadj, adjncy, w = graph_from_degrees(degs, rng, "lognormal", V=4096)
    if dist == "fewlights":      # almost every entry barely heavy, 1 % very light: a light tile spans many partners
        w = np.where(rng.random(len(w)) < 0.01, 0.01, 1.01).astype(np.float32)
    elif dist == "fewheavies":   # 0.1 % of the entries carry almost all the mass
        w = np.where(rng.random(len(w)) < 0.001, 1000.0, 0.5).astype(np.float32)
    else:
        w = weights(len(w), rng, dist)
    build_and_compare(orc, xadj, adjncy, w, "tiled/" + dist)


@pytest.mark.parametrize("dist", ["uniform", "lognormal2", "nearequal", "sparse", "fewlights", "fewheavies", "alternating"])
def test_rows_that_end_at_the_ends_of_wavefronts(orc, dist):
    # rows paired by a merge: the last wavefront full, one slot short, one slot into the next; every row start; lights or
    # heavies alone but for a few, which keeps one of the two sequences empty for whole wavefronts
    from helpers import weights
    from skywalker_amd import capi
    rng = np.random.default_rng(23)
    per = {253: (64, 4), 381: (64, 6), 509: (64, 8), 765: (128, 6), 1021: (128, 8), 1533: (256, 6), 2045: (256, 8),
           2557: (256, 10), 3069: (512, 6), 3581: (256, 14), 4093: (512, 8), 5117: (512, 10)}
    degs, lo = [], 193
    for hi, (threads, slots) in per.items():
        ends = [64 * slots * k + e for k in range(1, threads // 64 + 1) for e in (-1, 0, 1)]
        degs += [d for d in ends if lo <= d <= hi] + [lo, hi]
        lo = hi + 1
    degs += [1, 1, 2, 3] * 8
    rng.shuffle(degs)
    xadj, adjncy, w = graph_from_degrees(degs, rng, "lognormal", V=6000)
    if dist == "fewlights":
        w = np.where(rng.random(len(w)) < 0.01, 0.01, 1.01).astype(np.float32)
    elif dist == "fewheavies":
        w = np.where(rng.random(len(w)) < 0.005, 1000.0, 0.5).astype(np.float32)
    elif dist == "alternating":  # lights first, then heavies, then lights: the merge runs along one of them for long
        w = np.where((np.arange(len(w)) // 300) % 2 == 0, 1.0, 3.0).astype(np.float32)
    else:
        w = weights(len(w), rng, dist)
    build_and_compare(orc, xadj, adjncy, w, "ends/" + dist)
    g = capi.Graph.upload(xadj, adjncy, w)
    g.build_tables()
    compare_tables(orc, g, xadj, w, "ends in four launches/" + dist)
    g.free()


@pytest.mark.parametrize("dist", ["lognormal2", "nearequal", "sparse", "fewlights", "fewheavies", "alternating", "equal"])
def test_rows_that_share_a_wavefront(orc, dist):
    # rows of 3..192 entries, paired by a merge in strips of their own: every length a few times, so that full, partly filled
    # and empty strips meet; rows without heavies, with one, with nothing but heavies around one light
    from helpers import weights
    from skywalker_amd import capi
    rng = np.random.default_rng(29)
    degs = [d for d in range(1, 196) for _ in range(3)] + [8, 16, 32, 64, 128, 160, 192] * 20
    rng.shuffle(degs)
    xadj, adjncy, w = graph_from_degrees(degs, rng, "lognormal", V=len(degs) + 5)
    if dist == "fewlights":
        w = np.where(rng.random(len(w)) < 0.03, 0.01, 1.01).astype(np.float32)
    elif dist == "fewheavies":
        w = np.where(rng.random(len(w)) < 0.02, 1000.0, 0.5).astype(np.float32)
    elif dist == "alternating":
        w = np.where((np.arange(len(w)) // 20) % 2 == 0, 1.0, 3.0).astype(np.float32)
    else:
        w = weights(len(w), rng, dist)
    build_and_compare(orc, xadj, adjncy, w, "short/" + dist)
    g = capi.Graph.upload(xadj, adjncy, w)
    g.build_tables()
    compare_tables(orc, g, xadj, w, "short by default/" + dist)
    g.free()


def test_streaming_kernel_for_rows_with_too_many_tiles(orc):
    from skywalker_amd import capi
    rng = np.random.default_rng(22)
    xadj, adjncy, w = graph_from_degrees([4100, 9000, 20000, 3, 70000], rng, "lognormal2", V=4096)
    capi.set_option("tiled_max_tiles", 10)  # up to 9000 (9 tiles) stays tile-parallel, the other two are streamed
    try:
        build_and_compare(orc, xadj, adjncy, w, "streaming")
    finally:
        capi.set_option("tiled_max_tiles", 1 << 22)


def test_search_variant_of_the_row_kernels_gives_the_same_table(orc):
    # "row_merge" = 0 selects the kernels that do one binary search per entry (rows of 62..4093 entries) and
    # sends rows of 4094..5117 entries down the tile-parallel path (longer ones stream or go tile by tile anyway)
    from skywalker_amd import capi
    rng = np.random.default_rng(23)
    degs = [70, 126, 254, 300, 509, 510, 1021, 1500, 2046, 3000, 4093, 4094, 5000, 8189, 8190, 3, 0, 1]
    xadj, adjncy, w = graph_from_degrees(degs, rng, "lognormal", V=8192)
    capi.set_option("row_merge", 0)
    try:
        build_and_compare(orc, xadj, adjncy, w, "row_merge=0")
    finally:
        capi.set_option("row_merge", 1)
    build_and_compare(orc, xadj, adjncy, w, "row_merge=1")


@pytest.mark.parametrize("dist", ["lognormal2", "uniform", "nearequal", "sparse", "fewlights", "fewheavies"])
def test_rows_streamed_by_one_workgroup(orc, dist):
    # rows of 5118..8189 entries are held by one workgroup, its heavies listed in LDS (5632 at a time), rows of
    # 8190..524287 entries stream through one with a window of 5080 heavies ("fewlights" has rows with several lists
    # or windows, "uniform" too among the streamed ones, "nearequal" rows without a heavy); 524288 is the first degree
    # of the tile-parallel class
    from helpers import weights
    rng = np.random.default_rng(31)
    degs = [5118, 5119, 6000, 8189, 8190, 8191, 7, 8193, 12288, 2, 12289, 16381, 16382, 16385, 1, 30000, 65533, 65534, 0, 9001, 150001, 524287, 524288]
    xadj, adjncy, w = graph_from_degrees(degs, rng, "lognormal", V=4096)
    if dist == "fewlights":
        w = np.where(rng.random(len(w)) < 0.01, 0.01, 1.01).astype(np.float32)
    elif dist == "fewheavies":
        w = np.where(rng.random(len(w)) < 0.001, 1000.0, 0.5).astype(np.float32)
    else:
        w = weights(len(w), rng, dist)
    build_and_compare(orc, xadj, adjncy, w, "stream/" + dist)


@pytest.mark.parametrize("dist", ["lognormal2", "nearequal", "fewlights"])
def test_long_rows_that_end_at_the_ends_of_wavefronts(orc, dist):
    # held rows change hands in LDS by wavefronts of 1024 slots, streamed ones by quads of lanes where all 512 slots of a
    # wavefront are written and slot by slot elsewhere: ends at both sides of a wavefront's, of a quad's, every row start
    from helpers import weights
    rng = np.random.default_rng(37)
    degs = [1024 * k + e for k in (5, 6, 7) for e in (-1, 0, 1)] + [8 * 1024 - e for e in (5, 4, 3)]
    degs += [512 * k + e for k in (16, 17, 23, 24, 25, 32) for e in (-33, -4, -1, 0, 1, 2, 3, 31, 32)]
    degs = [d for d in degs if d >= 5118] + [1, 1, 2, 3] * 12
    rng.shuffle(degs)
    xadj, adjncy, w = graph_from_degrees(degs, rng, "lognormal", V=4096)
    w = np.where(rng.random(len(w)) < 0.01, 0.01, 1.01).astype(np.float32) if dist == "fewlights" else weights(len(w), rng, dist)
    build_and_compare(orc, xadj, adjncy, w, "ends of long rows/" + dist)


def test_special_weight_values_in_every_kind_of_row(orc):
    # NaN, infinities, negatives, -0, denormals, values at and beyond the 2^32 clamp, and values whose
    # contribution to the exact sum is only a few units of 2^-64: same bits as the oracle in every class
    rng = np.random.default_rng(41)
    degs = [1, 2, 3, 5, 9, 20, 40, 100, 150, 200, 400, 700, 1500, 3000, 5000, 6000, 8189, 9000, 20000, 70000]
    xadj, adjncy, w = graph_from_degrees(degs, rng, "lognormal", V=4096)
    special = np.array([np.nan, np.inf, -np.inf, -1.0, -0.0, 0.0, 1e-45, 1e-40, 2.0 ** -64, 2.0 ** -63, 3e-19,
                        2.0 ** 32, 2.0 ** 32 * 1.5, 3e38, 2.0 ** -20, 1.0, 123456.789], np.float32)
    pick = rng.random(len(w)) < 0.3
    w[pick] = special[rng.integers(0, len(special), pick.sum())]
    with np.errstate(all="ignore"):
        build_and_compare(orc, xadj, adjncy, w, "special values")
    # rows made of nothing but contributions that vanish: invalid rows in every class
    w2 = np.where(rng.random(len(w)) < 0.5, np.float32(1e-30), np.float32(-3.0)).astype(np.float32)
    build_and_compare(orc, xadj, adjncy, w2, "all-vanishing rows")


def test_build_profile_is_opt_in(orc):
    # without the option one bracket spans the build; with it every launched class has its own entry
    from skywalker_amd import capi
    g = capi.Graph.rmat(14, 16, 3, capi.W_UNIFORM, 1.0, 100.0, 3)
    sec = g.build_tables()
    prof = g.build_profile()
    assert [p[0] for p in prof] == ["build"] and prof[0][2] == g.E
    assert abs(prof[0][1] * 1e-3 - sec) < 1e-6
    before = g.tables()
    capi.set_option("build_profile", 1)
    try:
        sec = g.build_tables()
    finally:
        capi.set_option("build_profile", 0)
    prof = g.build_profile()
    assert prof[0][0] == "bin" and len(prof) > 3
    assert abs(sum(p[1] for p in prof) * 1e-3 - sec) < 1e-5  # the brackets tile the build
    after = g.tables()
    g.free()
    for a, b in zip(before, after):
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8))


def test_degenerate_inputs(orc):
    # a graph without edges, a graph without vertices, no walkers, zero steps: every entry point returns
    # cleanly and the counts are zero
    from skywalker_amd import capi
    for V in (0, 1, 300):
        xadj = np.zeros(V + 1, np.uint32)
        g = capi.Graph.upload(xadj, np.zeros(0, np.uint32), np.zeros(0, np.float32))
        assert g.V == V and g.E == 0
        g.build_tables()
        prob, alias, valid = g.tables()
        assert len(prob) == 0 and len(alias) == 0 and len(valid) == V and not valid.any()
        seeds = np.arange(min(V, 5), dtype=np.uint32)
        for length in (0, 4):
            p, l, sampled, _ = g.walk_offline(seeds, length, 0.0, 1)
            assert sampled == 0 and not l.to_host().any()
            assert np.array_equal(p.to_host((len(seeds), length + 1))[:, 0], seeds)
            p, l, sampled, _ = g.walk_online(capi.BIAS_STATIC, 1.0, 1.0, seeds, length, 0.0, 1)
            assert sampled == 0 and not l.to_host().any()
            p, l, sampled, _ = g.walk_online(capi.BIAS_NODE2VEC_REJECT, 2.0, 0.5, seeds, length, 0.0, 1)
            assert sampled == 0 and not l.to_host().any()
        d, sl, sampled, _ = g.sample_offline(seeds, [1, 3, 2], 1)
        assert sampled == 0 and not sl.to_host().any()
        d, sl, sampled, _ = g.sample_online(seeds, [1, 3, 2], 1)
        assert sampled == 0 and not sl.to_host().any()
        g.free()
    # an ordinary graph, no walkers
    xadj, adjncy = orc.rmat_csr(8, 4, 1)
    g = capi.Graph.upload(xadj, adjncy, None)  # unit weights
    g.build_tables()
    none = np.zeros(0, np.uint32)
    assert g.walk_offline(none, 5, 0.0, 1)[2] == 0
    assert g.walk_online(capi.BIAS_NODE2VEC, 2.0, 0.5, none, 5, 0.0, 1)[2] == 0
    assert g.sample_offline(none, [1, 2], 1)[2] == 0
    g.free()


@pytest.mark.parametrize("seed", range(8))
def test_random_mixtures_of_every_class(orc, seed):
    # both ends of every degree class plus random rows of every size, a different weight law per seed,
    # special values sprinkled into some
    from helpers import weights
    rng = np.random.default_rng(1000 + seed)
    ends = [0, 1, 2, 3, 5, 6, 8, 9, 13, 14, 16, 17, 29, 30, 32, 33, 61, 62, 64, 65, 125, 126, 128, 129, 191, 192, 193, 253, 254,
            381, 382, 509, 510, 765, 766, 5117, 5118, 8189, 8190, 16381, 16382, 24576, 24577, 65533, 65534]
    for nw in range(2, 11):
        ends += [512 * (nw - 1) - 2, 512 * nw - 3]
    degs = ends + list(rng.integers(0, 70, 3000)) + list(rng.integers(60, 600, 600)) + \
        list(rng.integers(500, 8300, 260)) + list(rng.integers(8000, 66000, 12)) + list(rng.integers(66000, 400000, 2))
    degs = np.array(degs)
    rng.shuffle(degs)
    xadj = np.zeros(len(degs) + 1, np.uint32)
    xadj[1:] = np.cumsum(degs)
    E = int(xadj[-1])
    adjncy = rng.integers(0, len(degs), E).astype(np.uint32)
    dist = ["lognormal", "uniform", "lognormal2", "nearequal", "sparse", "unit", "equal"][seed % 7]
    w = weights(E, rng, dist)
    if seed % 3 == 0:
        pick = rng.random(E) < 0.001
        special = np.array([0.0, -1.0, np.inf, np.nan, 1e-30, 2.0 ** -64, 2.0 ** 32, 1e38], np.float32)
        w[pick] = special[rng.integers(0, len(special), pick.sum())]
    with np.errstate(all="ignore"):
        build_and_compare(orc, xadj, adjncy, w, "mixture %d/%s" % (seed, dist))


def test_two_graphs_hold_different_settings(orc):
    # a knob set on one graph (sky_graph_set_option) leaves the other graph and the process-wide value alone
    from skywalker_amd import capi
    rng = np.random.default_rng(51)
    xadj, adjncy, w = graph_from_degrees(list(rng.integers(1, 200, 500)) + [300, 2000], rng, "lognormal")
    a = capi.Graph.upload(xadj, adjncy, w)
    b = capi.Graph.upload(xadj, adjncy, w)
    a.set_option("build_profile", 1)
    a.build_tables()
    b.build_tables()
    assert len(a.build_profile()) > 3 and [p[0] for p in b.build_profile()] == ["build"]
    c = capi.Graph.upload(xadj, adjncy, w)
    c.build_tables()
    assert [p[0] for p in c.build_profile()] == ["build"]  # the process-wide value did not move
    a.set_option("build_profile", None)
    a.build_tables()
    assert [p[0] for p in a.build_profile()] == ["build"]
    with pytest.raises(capi.SkyError):
        a.set_option("no_such_knob", 1)
    with pytest.raises(capi.SkyError):
        a.set_option("small_in_place", 7)
    want = a.tables()[0]
    for g in (a, b, c):
        assert np.array_equal(g.tables()[0], want)
        g.free()


def test_device_addresses_of_the_resident_arrays(orc):
    # sky_graph_device_ptrs: what lies at the addresses is what sky_graph_download and sky_alias_download give
    from skywalker_amd import capi
    import ctypes
    xadj, adjncy = orc.rmat_csr(10, 8, 5)
    w = orc.gen_weights(orc.W_UNIFORM, 5, len(adjncy), 1.0, 100.0)
    g = capi.Graph.upload(xadj, adjncy, w)
    g.build_tables()
    prob, alias, valid = g.tables()
    px, pa, pw, pt, pv = g.device_ptrs()
    assert px and pa and pw and pt and pv

    def read(addr, count, dtype):
        out = np.empty(count, dtype)
        capi._ck(capi.lib().sky_memcpy_d2h(capi._p(out), ctypes.c_void_p(addr), ctypes.c_size_t(out.nbytes)))
        return out
    assert np.array_equal(read(px, len(xadj), np.uint32), xadj)
    assert np.array_equal(read(pa, len(adjncy), np.uint32), adjncy)
    assert np.array_equal(read(pw, len(w), np.float32), w)
    entries = read(pt, 2 * len(w), np.uint32).reshape(-1, 2)  # {float prob; uint32 alias} per slot
    assert np.array_equal(entries[:, 0].view(np.float32), prob) and np.array_equal(entries[:, 1], alias)
    assert np.array_equal(read(pv, len(xadj) - 1, np.int8), valid)
    g.free()


def compare_tables(orc, g, xadj, w, label):
    oprob, oalias, ovalid = orc.alias_build(xadj, w)
    prob, alias, valid = g.tables()
    bad = np.flatnonzero((prob.view(np.uint32) != oprob.view(np.uint32)) | (alias != oalias))
    deg = np.diff(xadj)
    assert not len(bad), "%s: %d entries differ, first in a row of %d" % (
        label, len(bad), deg[np.searchsorted(xadj, bad[0], side="right") - 1])
    assert np.array_equal(valid, ovalid)


@pytest.mark.parametrize("stream_min_edges", [0, 4000000])
@pytest.mark.parametrize("dist", ["lognormal2", "uniform", "equal", "nearequal", "sparse"])
def test_builds_in_four_launches(orc, dist, stream_min_edges):
    # the default for up to 2^27 entries: rows of every class, those of 8190..65533 entries streamed or tile by tile; the
    # second and third build find the row lists of the first, with other weights and with the graph's own again
    from helpers import weights
    from skywalker_amd import capi
    rng = np.random.default_rng(51)
    degs = EDGE_DEGREES + [24576, 24577, 65533, 65534] + list(rng.integers(0, 300, 700)) + list(rng.integers(300, 9000, 40))
    rng.shuffle(degs)
    xadj, adjncy, w = graph_from_degrees(degs, rng, dist, V=len(degs) + 70)
    w2 = weights(len(w), rng, "sparse" if dist == "uniform" else "uniform")
    g = capi.Graph.upload(xadj, adjncy, w)
    g.set_option("stream_min_edges", stream_min_edges)
    g.build_tables()
    compare_tables(orc, g, xadj, w, dist)
    g.build_tables_from_weights(capi.DeviceArray.from_host(np.concatenate([w2, np.zeros(4, np.float32)])))
    compare_tables(orc, g, xadj, w2, dist + ", other weights")
    g.build_tables()
    compare_tables(orc, g, xadj, w, dist + ", again")
    g.free()


@pytest.mark.parametrize("n", [2047, 2048])
def test_many_rows_that_one_workgroup_holds(orc, n):
    # from 2,048 rows of 5,118..8,189 entries on they are a launch of their own behind the four
    rng = np.random.default_rng(47)
    degs = [5118, 5119, 8188, 8189] * (n // 4) + [6000] * (n % 4) + [12289, 1, 2, 3, 40, 700] + list(rng.integers(0, 40, 3000))
    rng.shuffle(degs)
    xadj, adjncy, w = graph_from_degrees(degs, rng, "lognormal", V=len(degs))
    w[xadj[100]:xadj[110]] = 0.0
    from skywalker_amd import capi
    g = capi.Graph.upload(xadj, adjncy, w)
    g.build_tables()
    compare_tables(orc, g, xadj, w, "held rows/%d" % n)
    g.free()


@pytest.mark.parametrize("longest", [509, 510, 12288, 12289])
@pytest.mark.parametrize("dist", ["lognormal2", "fewlights", "sparse"])
def test_small_builds_in_one_launch(orc, dist, longest):
    # rows of every class up to 12,288 entries share workgroups of 512 threads, a wavefront or a workgroup each; a longer row,
    # or none that needs more than a wavefront, takes the four launches; twice, the second time from weights without a row's
    from helpers import weights
    from skywalker_amd import capi
    rng = np.random.default_rng(43)
    degs = [d for d in EDGE_DEGREES if d < longest] + [longest] + list(rng.integers(0, min(longest, 2000), 300))
    rng.shuffle(degs)
    xadj, adjncy, w = graph_from_degrees(degs, rng, "lognormal", V=len(degs) + 3)
    w = np.where(rng.random(len(w)) < 0.01, 0.01, 1.01).astype(np.float32) if dist == "fewlights" else weights(len(w), rng, dist)
    g = capi.Graph.upload(xadj, adjncy, w)
    g.build_tables()
    compare_tables(orc, g, xadj, w, "one launch/%s/%d" % (dist, longest))
    g.free()
    for v in rng.integers(0, len(degs), 20):
        w[xadj[v]:xadj[v + 1]] = 0.0
    g = capi.Graph.upload(xadj, adjncy, w)
    g.build_tables()
    compare_tables(orc, g, xadj, w, "one launch, rows without weight/%s/%d" % (dist, longest))
    g.free()


@pytest.mark.parametrize("vertices", [1, 63, 64, 65, 32767, 32768, 32769])
@pytest.mark.parametrize("longest", [32, 510])
def test_short_rows_swept_by_class(orc, vertices, longest):
    # up to 32,768 vertices: a wavefront for every class of a range's rows (longest 32: the launch of single wavefronts, 510: the one
    # launch of eight); one more vertex: one wavefront for all of them.  Flags too: rows without entries and without weight
    from skywalker_amd import capi
    rng = np.random.default_rng(vertices + longest)
    degs = rng.integers(0, 33, vertices)
    degs[-1] = longest
    xadj, _, w = graph_from_degrees(degs, rng, "lognormal2", V=max(vertices, 2))
    w[rng.random(len(w)) < 0.3] = 0.0
    adjncy = np.zeros(len(w), np.uint32)
    g = capi.Graph.upload(xadj, adjncy, w)
    for _ in range(2):
        g.build_tables()
        compare_tables(orc, g, xadj, w, vertices)
    g.free()


def few_carry_the_mass(d, k0, e):
    """Shares of the mean weight, in units of 2^-40 all whole: one heavy, then lights whose deficits reach its surplus as the last
    of them is taken, e units more.  Deficits and surpluses together pass 2^53 on the way there for d > 4103, at an odd number."""
    u, n0 = 2.0 ** -40, d - 8
    share = np.zeros(d)
    share[:4] = [k0 * u, n0 + 4 - 2.0 ** -10, 1.5, (2 ** 30 - 2 ** 24) * u]
    share[4 + n0:] = [(2 ** 24 - k0 - e) * u, 2.0, 0.5 - 2.0 ** -20, (2 ** 20 + e) * u]
    w = share.astype(np.float32)
    assert np.array_equal(w.astype(np.float64), share) and share.sum() == d  # so that the scale is 1
    return w


def below_the_grid(d, k0, e):
    """The same meeting of a light and a heavy, d a power of two, with heavies between that add nothing to the row's sum (their
    weights are below 2^-64) and have a surplus of 0.75 d each: 0.6 d^2 altogether, past 2^53 units for d >= 128."""
    u, share = 2.0 ** -40, np.full(d, 0.25)
    h = d - d // 8
    share[:3] = [k0 * u, 3 - 2.0 ** -22, 1.5]
    share[3:h] = 0.75 * d
    share[3] = d  # a weight of 2^-64: the row's sum
    share[h] = (2 ** 18 - k0 - e) * u
    w = (share * (2.0 ** -64 / d)).astype(np.float32)
    assert np.array_equal(w.astype(np.float64), share * (2.0 ** -64 / d))
    return w


def skewed_rows():
    rows = [few_carry_the_mass(d, k0, e) for d in (3777, 4093, 4094, 4103, 4104, 4605, 4606, 5117) for k0 in (1, 3) for e in (-1, 0)]
    # in rows like these the last bit of one probability differed
    rows += [np.random.default_rng(s).lognormal(0, sigma, 5117).astype(np.float32) for s, sigma in ((49, 4), (2891, 3), (3448, 6))]
    rng = np.random.default_rng(61)
    return rows + [rng.lognormal(0, sigma, d).astype(np.float32) for sigma in (3, 4, 6) for d in rng.integers(3070, 5118, 20)]


def vanishing_rows():
    rows = [below_the_grid(d, k0, e) for d in (64, 128, 256, 512, 1024, 2048, 4096) for k0 in (1, 3, 5, 7) for e in (-1, 0)]
    rng, u = np.random.default_rng(62), 2.0 ** -64
    for d in [100, 128, 129, 192, 193, 381, 509, 765, 1021, 2045, 3069, 3581, 4093, 5117] + list(rng.integers(100, 5118, 20)):
        share = np.concatenate([1 + rng.uniform(0, 2.0 ** -19, d // 5), rng.uniform(0.5, 0.99, d // 2) * d,
                                rng.uniform(0, 0.001, d - d // 5 - d // 2)])
        share[d // 3] = d
        rows.append((share * (u / d)).astype(np.float32))
    return rows


def surpluses_that_leap(d, k, rng):
    """Heavies of a little surplus up to slot k, one light that all of them fall to, then forty heavies of some d / 3 shares each: the
    prefix of a thread that holds some of both kinds passes 2^53, what lies before it is a small odd number of units."""
    u, one = np.float32(2.0 ** -64), np.float32(3 * 2.0 ** -64 / d)  # one: the least heavy weight, or the largest light one
    w = (rng.uniform(0, 1, d) * one).astype(np.float32)
    w[0] = 0.0
    w[1:k] = one
    for i in range(1, k):
        for _ in range(1 + int(rng.integers(3))):
            w[i] = np.nextafter(w[i], np.float32(1))
    w[k:k + 40] = rng.uniform(0.9, 0.99, 40) * u
    w[k + 40] = 3 * u  # the row's sum
    return w


def leaping_rows():
    return [surpluses_that_leap(d, k, np.random.default_rng(k)) for d in (1021, 2557, 3100, 3581, 3800, 4093, 4094, 5117)
            for k in range(5, 30)]


@pytest.mark.parametrize("route", ["by class", "four launches", "one launch"])
@pytest.mark.parametrize("make", [skewed_rows, vanishing_rows, leaping_rows])
def test_rows_whose_sums_need_every_bit(orc, make, route):
    # rows whose deficits and surpluses together, or whose surpluses alone, add up to 2^53 units and more: the sums that decide
    # aliases and residuals are below that and exact in every kernel
    from skywalker_amd import capi
    rows = make()
    if route == "four launches":  # a row too long for one
        rows.append(np.ones(12289, np.float32))
    w = np.concatenate(rows)
    xadj = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.uint32)
    g = capi.Graph.upload(xadj, np.zeros(len(w), np.uint32), w)
    if route == "by class":
        g.set_option("small_in_place", 0)
    g.build_tables()
    compare_tables(orc, g, xadj, w, "%s, %s" % (make.__name__, route))
    g.free()


def long_vanishing_rows(longest):
    """Rows whose surpluses add up to 2^64 units and more."""
    rows = [below_the_grid(d, k0, e) for d in (8192, 16384, 65536) if d <= longest for k0 in (1, 3) for e in (-1, 0)]
    rng, u = np.random.default_rng(63), 2.0 ** -64
    for d in (5100, 5117, 5118, 6000, 8188, 8189, 8190, 9000, 12288, 12289, 30000, 70001, 600001):
        if d > longest:
            break
        share = np.concatenate([1 + rng.uniform(0, 2.0 ** -19, d // 10), rng.uniform(0.9, 0.99, d - 2 * (d // 10)) * d,
                                rng.uniform(0, 0.1, d // 10)])
        share[d // 3] = d
        rows.append((share * (u / d)).astype(np.float32))
    return rows


@pytest.mark.parametrize("longest", [12288, 600001])
@pytest.mark.parametrize("knobs", [{}, {"stream_min_edges": 0, "stream_wide_min_edges": 0}, {"small_in_place": 0},
                                   {"small_in_place": 0, "stream_min_edges": 0, "stream_wide_min_edges": 0}, {"row_merge": 0},
                                   {"tiled_max_tiles": 9}])
def test_surpluses_beyond_64_bits(orc, knobs, longest):
    # by default in one launch or four, streamed or tile by tile, by class (rows of 5,118..8,189 entries held), by the kernels that the
    # tests alone select
    from skywalker_amd import capi
    rows = long_vanishing_rows(longest)
    w = np.concatenate(rows)
    xadj = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.uint32)
    g = capi.Graph.upload(xadj, np.zeros(len(w), np.uint32), w)
    for k, value in knobs.items():
        g.set_option(k, value)
    g.build_tables()
    compare_tables(orc, g, xadj, w, "surpluses beyond 64 bits, %s" % knobs)
    g.free()


@pytest.mark.parametrize("walkers", [200, 1000, 5000])
def test_draws_from_rows_with_surpluses_beyond_64_bits(walkers):
    # evaluated from the weights, by workgroups of 256 and 128 threads, against those from the tables; 20 M entries in rows of 32 beside them
    from skywalker_amd import capi
    rows = long_vanishing_rows(12288)
    lens = np.concatenate([[len(r) for r in rows], np.full(625000, 32)])
    w = np.concatenate(rows + [np.ones(32 * 625000, np.float32)])
    xadj = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)
    local = np.arange(len(w), dtype=np.uint32) - np.repeat(xadj[:-1], lens)  # a vertex of its own for every slot of a row
    g = capi.Graph.upload(xadj, local, w)
    g.set_option("online_full_build", 0)
    g.set_option("online_direct", 1)  # no row is built
    seeds = np.arange(walkers, dtype=np.uint32) % len(rows)
    direct = [g.walk_online(capi.BIAS_STATIC, 1.0, 1.0, seeds, 1, 0.0, 5), g.walk_online(capi.BIAS_NODE2VEC, 2.0, 0.5, seeds, 1, 0.0, 5)]
    g.build_tables()
    tabled = g.walk_offline(seeds, 1, 0.0, 5)[0].to_host()
    for paths, _, _, _ in direct:
        assert np.array_equal(paths.to_host(), tabled)
    g.free()


@pytest.mark.parametrize("degree", [2048 * 1024 - 3, 2048 * 1024 + 1])
def test_ledger_of_rows_of_very_many_tiles_in_four_launches(orc, degree):
    # up to 2048 tiles every tile adds up its row's sums itself, above a launch in between does
    from helpers import weights
    from skywalker_amd import capi
    rng = np.random.default_rng(52)
    xadj = np.cumsum([0, 3, degree, 0, 700000, 5]).astype(np.uint32)
    adjncy = rng.integers(0, 5, int(xadj[-1]), dtype=np.uint32)
    w = weights(len(adjncy), rng, "sparse")
    g = capi.Graph.upload(xadj, adjncy, w)
    g.build_tables()
    compare_tables(orc, g, xadj, w, "row of %d" % degree)
    g.free()


def test_large_builds_leave_short_rows_in_place_and_reuse_their_lists(orc):
    # more than 2^27 entries: no four launches, and no binning once the first build has made the lists
    from helpers import weights
    from skywalker_amd import capi
    rng = np.random.default_rng(53)
    degs = np.concatenate([rng.integers(0, 12, (1 << 23) + 1), rng.integers(12, 700, 250000), rng.integers(700, 9000, 300),
                           [66001, 600001]])
    rng.shuffle(degs)
    xadj = np.concatenate([[0], np.cumsum(degs)]).astype(np.uint32)
    E = int(xadj[-1])
    assert E > 1 << 27
    g = capi.Graph.from_degrees(xadj, 7, capi.W_LOGNORMAL, 0.0, 1.0, 7)
    for seed in (0, 1):
        w = weights(E, np.random.default_rng(seed), "uniform")
        g.build_tables_from_weights(capi.DeviceArray.from_host(np.concatenate([w, np.zeros(4, np.float32)])))
        compare_tables(orc, g, xadj, w, "build %d" % seed)
    g.free()


@pytest.mark.parametrize("knobs", [{"row_merge": 0}, {"tiled_max_tiles": 9}, {"row_merge": 0, "tiled_max_tiles": 9}, {}])
@pytest.mark.parametrize("small_in_place", [-1, 0, 1])
def test_flags_follow_the_weights_of_the_latest_build(orc, knobs, small_in_place):
    # rows that had no weight in the build before, and rows uploaded as invalid, are valid again after a build from good
    # weights, whichever kernels build them and whether or not the build bins the vertices anew
    from helpers import weights
    from skywalker_amd import capi
    rng = np.random.default_rng(54)
    degs = EDGE_DEGREES + [10_000, 24577, 66000] + list(rng.integers(0, 300, 300))
    rng.shuffle(degs)
    xadj, adjncy, w = graph_from_degrees(degs, rng, "uniform")
    half = w.copy()
    for v in range(0, len(degs), 2):
        half[xadj[v]:xadj[v + 1]] = 0.0
    g = capi.Graph.upload(xadj, adjncy, w)
    for k, value in knobs.items():
        g.set_option(k, value)
    g.set_option("small_in_place", small_in_place)
    for seq, build in enumerate([np.zeros_like(w), w, half, w[::-1].copy(), half]):
        g.build_tables_from_weights(capi.DeviceArray.from_host(build))
        compare_tables(orc, g, xadj, build, "build %d with %s, small_in_place %d" % (seq, knobs, small_in_place))
    n = len(w)
    g.upload_tables(np.zeros(n, np.float32), np.full(n, capi.INVALID, np.uint32), np.zeros(len(degs), np.int8))
    g.build_tables()
    compare_tables(orc, g, xadj, w, "uploaded as invalid, %s, small_in_place %d" % (knobs, small_in_place))
    g.free()


@pytest.mark.parametrize("kind", ["build", "build by class", "walk", "walk on full tables", "sample", "session"])
def test_seconds_of_a_call_that_lists_the_rows_contain_the_listing(kind):
    # the first build on a graph, and the next one after a knob has changed how rows are built, lists the rows by class
    # (two passes over the row offsets).  Against the same call that finds the lists in place, the least of five times each:
    # at least as much longer as one pass over the offsets takes at 8 TB/s
    from skywalker_amd import capi
    V = 1 << 24
    xadj = np.arange(V + 1, dtype=np.uint32) * np.uint32(2)
    xadj[-1] += 40  # one row that is listed
    g = capi.Graph.from_degrees(xadj, 7, capi.W_UNIFORM, 1.0, 2.0, 7)
    seeds, one = (capi.DeviceArray.from_host(np.arange(n, dtype=np.uint32)) for n in (10, 1))
    g.set_option("small_in_place", 1 if kind == "build by class" else -1)
    g.set_option("online_full_build", 0 if kind == "walk" else -1)

    def call(listing=None):
        g.sample_session(np.zeros(0, np.uint32), [1, 2], 1)  # its begin leaves the graph without tables
        if listing:
            g.set_option("stream_min_edges", listing)
        if kind.startswith("build"):
            return g.build_tables()
        if kind == "walk":
            return g.walk_online(capi.BIAS_STATIC, 1.0, 1.0, seeds, 4, 0.0, 1)[3]
        if kind == "walk on full tables":  # a thousand steps of one walker: cheaper with every row built
            sec = g.walk_online(capi.BIAS_STATIC, 1.0, 1.0, one, 1000, 0.0, 1)[3]
            g.tables()
            return sec
        return (g.sample_online if kind == "sample" else g.sample_session)(seeds, [1, 2, 2], 1)[3]
    call()
    again, listing = min(call() for _ in range(5)), min(call(10 + k) for k in range(5))
    print(kind, "again %.1f us, with the listing %.1f us" % (again * 1e6, listing * 1e6))
    assert listing - again > 4 * V / 8e12
    g.free()


def test_rows_of_2558_to_3581_entries_beside_shorter_ones(orc):
    # enough of them for the launch of 256 threads, 14 slots each, in a build and in that of a frontier of more than 65,536 rows, whose
    # 700 streamed rows the workgroups ask for; the edges of their classes, and of those around them
    from skywalker_amd import capi
    rng = np.random.default_rng(59)
    degs = list(rng.integers(2558, 3582, 1400)) + [2556, 2557, 2558, 2559, 3069, 3070, 3071, 3580, 3581, 3582, 3583, 4093, 4094, 5117] * 3 + \
        list(rng.integers(8190, 12000, 650)) + list(rng.integers(8190, 65534, 50)) + [8190, 24576, 24577, 65533] + \
        list(rng.integers(1, 300, 3000)) + list(rng.integers(1, 4, 65000))
    rng.shuffle(degs)
    xadj, adjncy, w = graph_from_degrees(degs, rng, "lognormal")
    g = capi.Graph.upload(xadj, adjncy, w)
    g.set_option("stream_min_edges", 0)  # 50 rows of up to 65,533 entries would take as long as all others
    seeds = rng.permutation(len(degs)).astype(np.uint32)
    d, sl, sampled, _ = g.sample_online(seeds, [1, 2], 3)
    got = d.to_host(), sl.to_host()
    g.build_tables()
    prob, alias, valid = g.tables()
    g.free()
    oprob, oalias, ovalid = orc.alias_build(xadj, w)
    assert np.array_equal(prob.view(np.uint32), oprob.view(np.uint32)) and np.array_equal(alias, oalias) and np.array_equal(valid, ovalid)
    want = orc.sample_offline(xadj, adjncy, oprob, oalias, seeds, [1, 2], 3)
    assert np.array_equal(got[0], want[0].ravel()) and np.array_equal(got[1], want[1].ravel()) and sampled == want[2]


@pytest.mark.parametrize("V", [32769, 36863, 36864, 36865, 40959, 200001])
def test_short_rows_of_ranges_in_another_order(orc, V):
    # whole and partial groups of 64 ranges of vertices
    from skywalker_amd import capi
    rng = np.random.default_rng(V)
    degs = np.where(rng.random(V) < 0.02, rng.integers(33, 300, V), rng.integers(0, 34, V))
    xadj = np.concatenate([[0], np.cumsum(degs)]).astype(np.uint32)
    E = int(xadj[-1])
    adjncy = rng.integers(0, V, E, dtype=np.uint32)
    w = rng.lognormal(0, 1, E).astype(np.float32)
    w[rng.random(E) < 0.3] = 0.0
    g = capi.Graph.upload(xadj, adjncy, w)
    for _ in range(2):
        g.build_tables()
    prob, alias, valid = g.tables()
    g.free()
    oprob, oalias, ovalid = orc.alias_build(xadj, w)
    assert np.array_equal(prob.view(np.uint32), oprob.view(np.uint32)) and np.array_equal(alias, oalias) and np.array_equal(valid, ovalid)


@pytest.mark.parametrize("limit", [None, 0, 1 << 30])
@pytest.mark.parametrize("seeds_n", [3000, 70000])
def test_rows_of_8190_to_24576_entries_streamed_and_longer_ones_by_tiles(orc, seeds_n, limit):
    # or all of them streamed (limit 0), or none: in a build of all rows, in one of the longer rows for a walk, and in those of small
    # frontiers (all by tiles) and of large ones, of more than 65,536 rows, the streamed ones and those with tiles among them
    from skywalker_amd import capi
    rng = np.random.default_rng(61)
    degs = list(rng.integers(8190, 24577, 270)) + list(rng.integers(8190, 9000, 350)) + \
        [8189, 8190, 8191, 24576, 24577, 24578, 30000, 65533, 65534, 70001, 600001] + list(rng.integers(1, 200, 2000)) + [1, 2] * 34000
    rng.shuffle(degs)
    xadj, adjncy, w = graph_from_degrees(degs, rng, "lognormal2")
    # every vertex but a few, or the first ones and all long rows
    seeds = rng.permutation(len(degs))[:seeds_n] if seeds_n > 65536 else np.append(np.flatnonzero(np.diff(xadj) > 8000), np.arange(seeds_n))[:seeds_n]
    seeds = seeds.astype(np.uint32)
    oprob, oalias, ovalid = orc.alias_build(xadj, w)
    g = capi.Graph.upload(xadj, adjncy, w)
    g.set_option("online_full_build", 0)
    g.set_option("online_direct", 0)
    g.set_option("stream_min_edges", limit)
    d, sl, sampled, _ = g.sample_online(seeds, [1, 2, 2], 3)
    got = d.to_host(), sl.to_host()
    walk = g.walk_online(capi.BIAS_STATIC, 1.0, 1.0, seeds, 9, 0.0, 5)
    walked = walk[0].to_host(), walk[1].to_host()
    g.build_tables()
    prob, alias, valid = g.tables()
    g.free()
    assert np.array_equal(prob.view(np.uint32), oprob.view(np.uint32)) and np.array_equal(alias, oalias) and np.array_equal(valid, ovalid)
    want = orc.sample_offline(xadj, adjncy, oprob, oalias, seeds, [1, 2, 2], 3)
    assert np.array_equal(got[0], want[0].ravel()) and np.array_equal(got[1], want[1].ravel()) and sampled == want[2]
    paths, lengths, steps = orc.walk_offline(xadj, adjncy, oprob, oalias, seeds, 9, 0.0, 5)
    assert np.array_equal(walked[0], paths.ravel()) and np.array_equal(walked[1], lengths) and walk[2] == steps


@pytest.mark.parametrize("by_class", [False, True])
@pytest.mark.parametrize("longest", [600, 13000, 30000, 70001])
def test_builds_over_several_streams_one_after_another_and_from_two_threads(orc, longest, by_class):
    # the sweep and the long rows beside the other launches, a tile path among these for the longest (rows of up to 600 entries are
    # one launch), or the class kernels on four streams: two weight arrays in turn, so that what an earlier build left shows, written
    # just before each build and read just after it; two graphs, a thread each
    import threading
    from helpers import weights
    from skywalker_amd import capi
    made, errors = [], []
    for k in range(2):
        rng = np.random.default_rng(longest + k)
        degs = np.concatenate([rng.integers(0, 33, 40000), rng.integers(33, 510, 4000), rng.integers(510, min(longest, 6000) + 1, 1500),
                               rng.integers(min(longest, 8190), longest + 1, 12), [longest]])
        rng.shuffle(degs)
        xadj, adjncy, w = graph_from_degrees(degs, rng, "lognormal")
        sets = [w, weights(len(w), rng, "lognormal2")]
        made.append((capi.Graph.upload(xadj, adjncy, w), sets, [orc.alias_build(xadj, x) for x in sets]))
        if by_class:
            made[k][0].set_option("small_in_place", k)

    def builds(g, sets, want):
        try:
            for n in range(6):
                x = capi.DeviceArray.from_host(np.concatenate([sets[n % 2], np.zeros(4, np.float32)]))
                g.build_tables_from_weights(x)
                prob, alias, valid = g.tables()
                oprob, oalias, ovalid = want[n % 2]
                assert np.array_equal(prob.view(np.uint32), oprob.view(np.uint32)) and np.array_equal(alias, oalias), n
                assert np.array_equal(valid, ovalid), n
        except BaseException as e:  # a thread's failure is the test's
            errors.append(e)
    builds(*made[0])
    threads = [threading.Thread(target=builds, args=m) for m in made]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for g, _, _ in made:
        g.free()
    if errors:
        raise errors[0]


@pytest.mark.parametrize("E", [(1 << 24) - 1, 1 << 24])
@pytest.mark.parametrize("longer", [False, True])
def test_rows_of_2558_to_5117_entries_in_a_launch_of_their_own(orc, E, longer):
    # the smallest build that gives them one and the largest that does not; the edges of their classes; enough rows of 2558..3581 entries that
    # these go out with the launch of 256 threads.  A row of more than 12288 entries keeps the build out of the one launch of small ones.
    from skywalker_amd import capi
    rng = np.random.default_rng(61)
    degs = list(rng.integers(2558, 5118, 300)) + [2557, 2558, 3069, 3070, 3581, 3582, 4093, 4094, 4605, 4606, 5117, 5118] * 2 + \
        list(rng.integers(1, 300, 20000)) + list(rng.integers(8190, 9000, 20)) + [13000] + list(rng.integers(2558, 3582, 1500 if longer else 0))
    left = E - sum(degs)
    degs += [31] * (left // 31) + [left % 31]
    rng.shuffle(degs)
    xadj = np.concatenate([[0], np.cumsum(degs)]).astype(np.uint32)
    adjncy = np.zeros(E, np.uint32)
    w = rng.lognormal(0, 2, E).astype(np.float32)
    g = capi.Graph.upload(xadj, adjncy, w)
    # a graph's first build goes out in order where there are no side streams yet; from other weights, so that rows the second leaves out show
    g.build_tables_from_weights(capi.DeviceArray.from_host(np.concatenate([w[::-1], np.zeros(4, np.float32)])))
    g.build_tables()
    prob, alias, valid = g.tables()
    g.free()
    oprob, oalias, ovalid = orc.alias_build(xadj, w)
    assert np.array_equal(prob.view(np.uint32), oprob.view(np.uint32)) and np.array_equal(alias, oalias) and np.array_equal(valid, ovalid)
