"""Dense table apply and the threshold ("DCT") codec on the GPU against the oracle.

Known answers come from the reference's own tests: dense pull round trip and SGD
(kraken/test/worker/emitter_test.cc:36-63), Abs/TopK/Take/ToCoo/ToDense/LtKeep vectors
(kraken/test/t/math_test.cc:323-382).
"""
import numpy as np
import pytest

from util import OPTIM_CASES, STATE_OF, assert_close, make_optims

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def api():
    from kraken_amd import api as a
    a.lib()
    return a


def test_dense_roundtrip_and_sgd(api, oracle):
    rng = np.random.default_rng(0)
    d0 = rng.standard_normal((10, 10)).astype(np.float32)
    g0 = rng.standard_normal((10, 10)).astype(np.float32)
    t = api.DenseTable(d0)
    rc, r0 = t.Pull()
    assert rc == 0 and np.array_equal(r0, d0.ravel())            # emitter_test.cc:36-49
    lr = 0.37
    assert t.Push(api.Optim.create(api.OptimType.kSGD), g0, lr) == 0
    assert np.array_equal(t.Pull()[1], (d0 - np.float32(lr) * g0).ravel())   # :51-63
    assert t.Push(api.Optim.create(api.OptimType.kSGD), g0.ravel()[:7], lr) == 11


@pytest.mark.parametrize("name,type_,conf", OPTIM_CASES, ids=[c[0] for c in OPTIM_CASES])
@pytest.mark.parametrize("n", [1000, 150_000, 4099])
def test_dense_optimizers_match_oracle(api, oracle, name, type_, conf, n):
    rng = np.random.default_rng(n + type_)
    w0 = rng.standard_normal(n).astype(np.float32)
    t = api.DenseTable(w0)
    r = oracle.DenseTable(w0)
    o_ref, o_gpu = make_optims(oracle, api, type_, conf)
    for step in range(5):
        g = (rng.standard_normal(n) * 1e-3).astype(np.float32)
        assert t.Push(o_gpu, g, 0.01) == 0
        assert r.push(o_ref, g, 0.01) == 0
    assert_close(t.Pull()[1], r.pull(), name)
    for st in STATE_OF[type_]:
        want = r.state(st)
        got = t.state(st)
        assert_close(got, want if want is not None else np.zeros(n, np.float32), "%s state %d" % (name, st))
    if type_ == 1:
        assert t.steps == r.steps == 5


def test_dense_coo_push(api, oracle):
    rng = np.random.default_rng(5)
    n = 20_000
    w0 = rng.standard_normal(n).astype(np.float32)
    g = rng.standard_normal(n).astype(np.float32)
    idx, val = oracle.to_coo(g, 1.0)
    for type_, conf in ((1, {}), (0, {}), (3, {"momentum": 0.9}), (2, {"centered": True})):
        t = api.DenseTable(w0)
        r = oracle.DenseTable(w0)
        o_ref, o_gpu = make_optims(oracle, api, type_, conf)
        for _ in range(3):
            assert t.PushCoo(o_gpu, idx, val, 0.01) == 0
            assert r.push_coo(o_ref, idx, val, 0.01) == 0
        assert_close(t.Pull()[1], r.pull(), "coo push type %d" % type_)
        # an empty COO gradient changes nothing, not even Adam's step counter (adam.cc:26-29)
        before = t.Pull()[1]
        assert t.PushCoo(o_gpu, np.zeros(0, np.int64), np.zeros(0, np.float32), 0.01) == 0
        assert np.array_equal(t.Pull()[1], before)
        if type_ == 1:
            assert t.steps == 3
    # repeated indices add up (t/math.cc:1043)
    t = api.DenseTable(np.zeros(8, np.float32))
    assert t.PushCoo(api.Optim.create(api.OptimType.kSGD), [3, 3, 5], [1.0, 2.0, 4.0], 1.0) == 0
    assert np.array_equal(t.Pull()[1], np.float32([0, 0, 0, -3, 0, -4, 0, 0]))


KAT10 = np.array([-1.0, 1.0, 2.0, 3.0, -4.0, -0.1, 0.001, 0.00001, 0.000001, 128], np.float32)


def test_coo_to_dense_known_answer(api, oracle):
    """math_test.cc:356-370: ToCoo(0.01) -> ToDense."""
    idx, val = oracle.to_coo(KAT10, 0.01)
    dense = api.coo_to_dense(idx, val, 10)
    assert np.array_equal(dense, np.float32([-1.0, 1.0, 2.0, 3.0, -4.0, -0.1, 0, 0, 0, 128]))
    assert np.array_equal(api.coo_to_dense([3, 3, 5], [1.0, 2.0, 4.0], 8),
                          np.float32([0, 0, 0, 3, 0, 4, 0, 0]))


def test_codec_small_passthrough(api):
    bag = api.DenseBag(100)
    assert bag.MaybeToCoo(1000, 0.75, np.ones(100, np.float32)) == (None, None)
    assert bag.step == 0


@pytest.mark.parametrize("n", [256, 4096, 65_536, 1_000_003])
@pytest.mark.parametrize("eta", [0.5, 0.75, 0.9])
def test_codec_matches_oracle(api, oracle, n, eta):
    """Three consecutive steps with life_span 2: a re-select, a stale-threshold step, a
    re-select; indices, values, threshold and residual all exact."""
    rng = np.random.default_rng(n)
    bag = api.DenseBag(n)
    ref = oracle.DctState(n)
    for step in range(3):
        g = rng.standard_normal(n).astype(np.float32)
        if step == 1:
            m = g[1::3].size
            g[::3][:m] = g[1::3]                   # ties around the threshold
        idx, val = bag.MaybeToCoo(2, eta, g)
        ridx, rval = ref.compress(g, life_span=2, eta=eta, exact_select=True)
        assert bag.tau == ref.tau
        assert np.array_equal(idx, ridx) and np.array_equal(val, rval)
        assert np.array_equal(bag.residual, ref.residual)
        if step % 2 == 0:
            assert idx.size >= int(n * (1.0 - eta))
    assert bag.step == ref.step == 3
    # decode(coo) + residual == corrected gradient, exactly
    dense = api.coo_to_dense(idx, val, n)
    assert np.array_equal(dense, oracle.coo_to_dense(ridx, rval, n))


def test_codec_reference_chunked_topk_agrees_when_chunks_divide(api, oracle):
    """The reference's TopK splits the tensor into t_num chunks and drops n mod t_num trailing
    elements (t/math.cc:573-586). When t_num divides n its threshold is the true k-th largest,
    which is what the GPU computes."""
    n = 8192
    rng = np.random.default_rng(3)
    g = rng.standard_normal(n).astype(np.float32)
    bag = api.DenseBag(n)
    ref = oracle.DctState(n)
    idx, val = bag.MaybeToCoo(1000, 0.75, g)
    ridx, rval = ref.compress(g, life_span=1000, eta=0.75, hw_threads=4, exact_select=False)
    assert bag.tau == ref.tau and np.array_equal(idx, ridx) and np.array_equal(val, rval)


def test_codec_device_pointers_and_capacity(api, oracle):
    n = 300_000
    rng = np.random.default_rng(8)
    g = rng.standard_normal(n).astype(np.float32)
    bag = api.DenseBag(n)
    small_i = np.empty(10, np.int64)
    small_v = np.empty(10, np.float32)
    with pytest.raises(api.KrakenHipError) as e:
        bag.MaybeToCoo(1000, 0.75, g, small_i, small_v)
    assert e.value.code == api.E_CAPACITY and bag.step == 0     # nothing was committed
    d_g = api.DeviceArray.from_host(g)
    d_idx, d_val, nnz = bag.MaybeToCoo(1000, 0.75, d_g)
    ref = oracle.DctState(n)
    ridx, rval = ref.compress(g, exact_select=True)
    assert nnz == ridx.size
    assert np.array_equal(d_idx.to_host()[:nnz], ridx) and np.array_equal(d_val.to_host()[:nnz], rval)
    assert np.array_equal(bag.residual, ref.residual)


@pytest.mark.parametrize("n", [256, 8191, 8192, 8193, 600_001, 9_000_001])
@pytest.mark.parametrize("eta", [0.02, 0.75, 0.99])
def test_codec_single_pass_emit(api, oracle, n, eta):
    """Device buffers with room for everything: one pass emits. One tile, tiles' edges, more tiles
    than workgroups, tiles that keep everything or nothing; three steps on one codec (the tiles'
    announcements of one step must not be taken for the next one's)."""
    rng = np.random.default_rng(n)
    bag, ref = api.DenseBag(n), oracle.DctState(n)
    for step in range(3):
        g = rng.standard_normal(n).astype(np.float32)
        d_idx, d_val, nnz = bag.MaybeToCoo(2, eta, api.DeviceArray.from_host(g))
        ridx, rval = ref.compress(g, life_span=2, eta=eta, exact_select=True)
        assert nnz == ridx.size, step
        assert np.array_equal(d_idx.to_host()[:nnz], ridx) and np.array_equal(d_val.to_host()[:nnz], rval), step
        assert np.array_equal(bag.residual, ref.residual), step
    bag.close()


@pytest.mark.parametrize("n", [4095, 4096, 4097, 1 << 19, (1 << 19) + 1, 8192 * 256, 8192 * 256 + 1, 16384 * 2048 + 1])
def test_codec_single_pass_tile_sizes(api, n):
    """Where the tiles' size changes (2^19 and 2^25 elements), at their edges, and with as many tiles as workgroups and
    one more: the pairs, in order, and the residual, against numpy with the threshold that the codec found."""
    rng = np.random.default_rng(n)
    bag = api.DenseBag(n)
    e = np.zeros(n, np.float32)
    for step in range(2):
        g = rng.standard_normal(n, dtype=np.float32)
        d_idx, d_val, nnz = bag.MaybeToCoo(2, 0.75, api.DeviceArray.from_host(g))
        f = g + e
        a = np.abs(f)
        if step == 0:                                # the k-th largest of k = n / 4
            assert bag.tau == np.partition(a, n - int(n * 0.25))[n - int(n * 0.25)]
        idx = np.flatnonzero(a >= bag.tau)
        assert nnz == idx.size
        assert np.array_equal(d_idx.to_host()[:nnz], idx) and np.array_equal(d_val.to_host()[:nnz], f[idx])
        e = np.where(a < bag.tau, f, np.float32(0))
        assert np.array_equal(bag.residual, e)
    bag.close()


@pytest.mark.parametrize("case", ["sgd_mom", "adam_amsgrad", "rmsprop_all"])
@pytest.mark.parametrize("n", [(1 << 22), (1 << 22) + 2049])
def test_dense_push_coo_tiles(api, oracle, case, n):
    """The tile-by-tile update with every number of state columns: ascending indices with empty tiles,
    a single entry, then unordered ones, blocking and asynchronous."""
    _, type_, conf = next(c for c in OPTIM_CASES if c[0] == case)
    from util import make_optims
    rng = np.random.default_rng(n)
    w0 = rng.standard_normal(n).astype(np.float32)
    t, r = api.DenseTable(w0), oracle.DenseTable(w0)
    o_ref, o_gpu = make_optims(oracle, api, type_, conf)
    ascending = np.sort(rng.choice(n // 2, size=n // 8, replace=False)).astype(np.int64) + n // 4
    for flags in (api.DEVICE_PTRS, api.DEVICE_PTRS | api.ASYNC):
        for idx in (ascending, np.array([n - 1], np.int64), ascending[::-1].copy()):
            val = (rng.integers(1, 65, size=idx.size) / 1024.0).astype(np.float32)
            d_idx, d_val = api.DeviceArray.from_host(idx), api.DeviceArray.from_host(val)
            assert api.lib().krk_dense_push_coo(t.h, api.C.byref(o_gpu.raw), api.C.c_void_p(d_idx.ptr),
                                                api.C.c_void_p(d_val.ptr), idx.size, 0.01, flags) == 0
            assert r.push_coo(o_ref, idx, val, 0.01) == 0
            assert_close(t.Pull()[1], r.pull(), "%d entries" % idx.size)


@pytest.mark.parametrize("n", [1 << 22, (1 << 22) + 1, 5_000_003])
def test_coo_to_dense_large_tensors(api, oracle, n):
    """From 2^22 elements on the dense result is written tile by tile when the indices ascend
    strictly (what ToCoo produces); anything else is zeroed and scattered into. Both against the
    oracle: ascending with long gaps and a full last tile, every element present, nothing present,
    shuffled, with repeats (which add up, t/math.cc:1043)."""
    rng = np.random.default_rng(n)

    def check(idx, val):
        idx = np.ascontiguousarray(idx, np.int64)
        val = np.ascontiguousarray(val, np.float32)
        want = np.zeros(n, np.float32)
        np.add.at(want, idx, val)
        if np.unique(idx).size == idx.size:
            assert np.array_equal(want, oracle.coo_to_dense(idx, val, n))
        assert np.array_equal(api.coo_to_dense(idx, val, n), want)
        d = api.coo_to_dense(api.DeviceArray.from_host(idx), api.DeviceArray.from_host(val), n)
        assert np.array_equal(d.to_host(), want)

    quarter = np.sort(rng.choice(n, size=n // 4, replace=False))
    check(quarter, rng.standard_normal(quarter.size))
    few = np.array([0, 5, 4095, 4096, n - 4097, n - 1])          # empty tiles in between, both ends
    check(few, rng.standard_normal(few.size))
    check(np.arange(n), rng.standard_normal(n))                   # every element
    check(np.zeros(0, np.int64), np.zeros(0, np.float32))         # nothing
    check(rng.permutation(quarter), rng.standard_normal(quarter.size))          # not ascending
    twice = np.sort(np.concatenate([quarter[:1000], quarter[:1000], quarter[5000:6000]]))
    check(twice, (rng.integers(-8, 9, size=twice.size) / 8.0))    # repeats add up (exact sums)
    # device indices that start 8 bytes into a 16-byte unit (a view into a larger buffer)
    import ctypes as C
    val = rng.standard_normal(quarter.size).astype(np.float32)
    shifted = api.DeviceArray.from_host(np.concatenate([[0], quarter]).astype(np.int64))
    d_val = api.DeviceArray.from_host(val)
    out = api.DeviceArray(n, np.float32)
    rc = api.lib().krk_coo_to_dense(C.c_void_p(shifted.ptr + 8), C.c_void_p(d_val.ptr), quarter.size,
                                    C.c_void_p(out.ptr), n, api.DEVICE_PTRS)
    assert rc == 0
    want = np.zeros(n, np.float32)
    want[quarter] = val
    assert np.array_equal(out.to_host(), want)


@pytest.mark.parametrize("idx", [[-6000, -5000], [-(1 << 40), -(1 << 39), 3], [-3, -2, -1, 0, 2047, 2048],
                                 [5, 1 << 22, (1 << 22) + 1], [1 << 40, (1 << 40) + 1], [-1, (1 << 22) - 1]],
                         ids=["below", "far_below", "around_zero", "around_n", "far_above", "ends"])
def test_coo_indices_outside_a_large_tensor(api, oracle, idx):
    """Entries outside [0, n) are skipped, also where they ascend, and nothing is written for them: not
    the tiles' starts either, which a negative entry behind another one named before the array."""
    n = 1 << 22
    idx = np.array(idx, np.int64)
    val = np.arange(1, idx.size + 1, dtype=np.float32)
    want = np.zeros(n, np.float32)
    inside = (idx >= 0) & (idx < n)
    want[idx[inside]] = val[inside]
    assert np.array_equal(api.coo_to_dense(idx, val, n), want)
    w0 = np.ones(n, np.float32)
    t = api.DenseTable(w0)
    opt = api.Optim.create(api.OptimType.kSGD)
    for _ in range(2):
        assert t.PushCoo(opt, idx, val, 0.5) == 0
        w0 = w0 - np.float32(0.5) * want
        assert np.array_equal(t.Pull()[1], w0)


def test_coo_gaps_of_every_length(api, oracle):
    """Empty tiles before, between and behind the entries: gaps that a lane fills alone, that it just no
    longer does and that take a wavefront several rounds, several of them in one wavefront."""
    n, tile = (1 << 23) + 5, 2048
    tiles = -(-n // tile)
    gaps = [0, 1, 7, 8, 9, 10, 63, 64, 65, 129, 0, 0, 8, 9]
    starts = np.cumsum(gaps)
    cases = [[0], [n - 1], [0, n - 1], [7 * tile], [8 * tile], [9 * tile], list(starts * tile + 3),
             list(range(300)), list(range(n - 300, n)), list(range(40 * tile, 40 * tile + 129)),
             [(tiles - 9) * tile - 1], [(tiles - 8) * tile - 1], [(tiles - 10) * tile]]
    for entries in cases:
        idx = np.unique(np.array(entries, np.int64))
        val = np.arange(1, idx.size + 1, dtype=np.float32)
        want = np.zeros(n, np.float32)
        want[idx] = val
        assert np.array_equal(api.coo_to_dense(idx, val, n), want), entries[:4]


def _many_entries(case, n):
    """Ascending indices, an entry in eight elements or more."""
    rng = np.random.default_rng(7)
    if case == "front":                  # one long run of entries and nothing behind it
        return np.arange(n // 6)
    if case == "back":
        return np.arange(n - n // 6, n)
    if case == "tiles":                  # every third tile full, the first and the last of the others' elements too
        i = np.arange(n)
        t, at = i // 2048, i % 2048
        return i[(t % 3 == 0) | ((t % 3 == 1) & ((at == 0) | (at == 2047)))]
    if case == "gaps":                   # stretches of a few words with gaps of 1 to 200 words between them
        size, gap = rng.integers(1, 40, n // 32) * 32 + rng.integers(0, 32, n // 32), rng.integers(1, 200, n // 32) * 32
        at = np.cumsum(size + gap) - size
        i = np.concatenate([np.arange(a, a + s) for a, s in zip(at[at < n], size)])
        return i[i < n]
    keep = rng.random(n) < dict(half=0.5, fifth=0.2, all=2.0)[case]
    return np.flatnonzero(keep)


@pytest.mark.parametrize("n", [1 << 22, (1 << 22) + 2047])
@pytest.mark.parametrize("case", ["front", "back", "tiles", "gaps", "half", "fifth", "all"])
def test_coo_many_entries(api, oracle, case, n):
    """Tensors with an entry in eight elements or more: decode and push, every element exact. Then with the number of
    entries next to where a wavefront's chunks and runs of chunks end, and with one pair out of order, one
    index twice and one outside, where two wavefronts meet."""
    full = _many_entries(case, n).astype(np.int64)
    assert full.size * 8 >= n
    t = api.DenseTable(np.zeros(n, np.float32))
    opt = api.Optim.create(api.OptimType.kSGD)
    w = np.zeros(n, np.float32)

    def check(idx):
        nonlocal w
        val = (np.arange(idx.size) % 61 - 30).astype(np.float32)
        inside = (idx >= 0) & (idx < n)
        want = np.zeros(n, np.float32)
        np.add.at(want, idx[inside], val[inside])
        assert np.array_equal(api.coo_to_dense(idx, val, n), want)
        assert t.PushCoo(opt, idx, val, 0.5) == 0
        w = w - np.float32(0.5) * want
        assert np.array_equal(t.Pull()[1], w)

    check(full)
    for cut in (1, 31, 32, 255, 256, 257, 1023, 1024, 1025):
        check(full[full.size % 1024 + 1024 - cut:] if case == "back" else full[:full.size - full.size % 1024 - 1024 + cut])
    at = full.size // 2 // 1024 * 1024
    swapped, twice, outside = full.copy(), full.copy(), full.copy()
    swapped[[at - 1, at]] = swapped[[at, at - 1]]
    twice[at] = twice[at - 1]
    outside[-1] = n
    for idx in (swapped, twice, outside):
        check(idx)
    check(full)


@pytest.mark.parametrize("case", ["front", "back", "tiles", "gaps", "fifth"])
def test_coo_decode_of_millions_of_entries(api, case):
    """Decodes leave a bit an element from 7 * 2^18 entries on: just below that and just above, and all of them."""
    n = 14_000_001                                     # (an entry in eight elements is less than that)
    full = _many_entries(case, n).astype(np.int64)
    assert n < 8 * ((7 << 18) - 1) and full.size > (7 << 18) + 1
    for count in ((7 << 18) - 1, 7 << 18, (7 << 18) + 1, full.size):
        idx = full[:count]
        val = (np.arange(count) % 61 - 30).astype(np.float32)
        want = np.zeros(n, np.float32)
        want[idx] = val
        assert np.array_equal(api.coo_to_dense(idx, val, n), want)


def test_dense_push_coo_large(api, oracle):
    n = (1 << 22) + 77
    rng = np.random.default_rng(4)
    w0 = rng.standard_normal(n).astype(np.float32)
    t, r = api.DenseTable(w0), oracle.DenseTable(w0)
    from util import make_optims
    o_ref, o_gpu = make_optims(oracle, api, 1, {})
    for step in range(3):
        idx = np.sort(rng.choice(n, size=n // 5, replace=False)).astype(np.int64)
        if step == 2:
            idx = rng.permutation(idx)                            # the scatter path
        val = (rng.integers(-64, 65, size=idx.size) / 1024.0).astype(np.float32)
        assert t.PushCoo(o_gpu, idx, val, 0.01) == 0 and r.push_coo(o_ref, idx, val, 0.01) == 0
        assert_close(t.Pull()[1], r.pull(), "step %d" % step)
    # an entry outside [0, n) is skipped, the others are applied
    bad = np.array([0, n], np.int64)
    one = np.ones(2, np.float32)
    assert t.PushCoo(o_gpu, bad, one, 0.01) == 0 and r.push_coo(o_ref, bad[:1], one[:1], 0.01) == 0
    assert_close(t.Pull()[1], r.pull(), "after an out-of-range entry")


_GROUP_CASES = [c for c in OPTIM_CASES if c[0] in ("sgd_mom", "adagrad_wd", "adam", "adam_amsgrad", "rmsprop_all")]


@pytest.mark.parametrize("name,type_,conf", _GROUP_CASES, ids=[c[0] for c in _GROUP_CASES])
def test_dense_group_matches_the_per_table_loop(api, oracle, name, type_, conf):
    """Ps::CombinePullDenseTable (ps/ps_op.cc:177-252) and a step's PushDenseTable calls for every
    dense parameter of a model, as one launch each: against the oracle's loop over the tables.
    Member sizes put some members off the 16-byte grid of the concatenated arrays (the scalar
    path), one member is empty, and a member that was updated on its
    own before joining keeps its own Adam step count."""
    rng = np.random.default_rng(type_ + 40)
    sizes = [64, 1, 150_000, 4099, 0, 7, 1024, 333] + [int(x) for x in rng.integers(1, 3000, size=32)]
    w0 = [rng.standard_normal(n).astype(np.float32) for n in sizes]
    tables = [api.DenseTable(w) for w in w0]
    refs = [oracle.DenseTable(w) for w in w0]
    o_ref, o_gpu = make_optims(oracle, api, type_, conf)
    g = (rng.standard_normal(sizes[2]) * 1e-3).astype(np.float32)
    assert tables[2].Push(o_gpu, g, 0.01) == 0 and refs[2].push(o_ref, g, 0.01) == 0
    grp = api.DenseGroup(tables)
    assert grp.n == sum(sizes)
    for step in range(3):
        grads = (rng.standard_normal(grp.n) * 1e-3).astype(np.float32)
        assert grp.CombinePush(o_gpu, grads, 0.01) == 0
        at = 0
        for r, n in zip(refs, sizes):
            if n:
                assert r.push(o_ref, grads[at:at + n], 0.01) == 0
            at += n
        if step == 1:    # a member's own call in between is ordered with the group's
            g = (rng.standard_normal(sizes[3]) * 1e-3).astype(np.float32)
            assert tables[3].Push(o_gpu, g, 0.01) == 0 and refs[3].push(o_ref, g, 0.01) == 0
    rc, got = grp.CombinePull()
    assert rc == 0
    want = np.concatenate([r.pull() for r in refs])
    assert_close(got, want, name + " combined pull")
    for t, r, n in zip(tables, refs, sizes):
        if n:
            assert np.array_equal(t.Pull()[1], got[sum(sizes[:tables.index(t)]):][:n])
            for st in STATE_OF[type_]:
                ws = r.state(st)
                assert_close(t.state(st), ws if ws is not None else np.zeros(n, np.float32), "%s state %d" % (name, st))
    if type_ == 1:
        assert [t.steps for t in tables if t.n] == [r.steps for r, n in zip(refs, sizes) if n]
        assert tables[2].steps == 4 and tables[3].steps == 4
    # the wrong total is the reference's code 11; device pointers work the same way
    assert grp.CombinePush(o_gpu, np.zeros(grp.n - 1, np.float32), 0.01) == 11
    d_out = api.DeviceArray(grp.n, np.float32)
    assert grp.CombinePull(out=d_out, async_=True)[0] == 0 and grp.sync() == 0
    assert np.array_equal(d_out.to_host(), got)
    grp.close()
    assert tables[0].Pull()[0] == 0       # members work on their own again


# a push takes 64 members a launch; columns are created by the group's push (200 a launch enter its
# descriptors), by a member's own while the group is there, and before the group
@pytest.mark.parametrize("members", [1, 64, 65, 130])
def test_dense_group_members_and_columns(api, oracle, members):
    rng = np.random.default_rng(members)
    sizes = [int(x) for x in rng.integers(1, 1500, size=members)]
    sizes[members // 2] = sizes[-1] = 0
    if members == 1:
        sizes = [1031]
    w0 = [rng.standard_normal(n).astype(np.float32) for n in sizes]
    tables, refs = [api.DenseTable(w) for w in w0], [oracle.DenseTable(w) for w in w0]
    own = 0
    for optims in (("adagrad", "adam"), ("sgd_mom", "adam")):
        grp = api.DenseGroup(tables)
        for name in optims:
            type_, conf = next(c[1:] for c in OPTIM_CASES if c[0] == name)
            o_ref, o_gpu = make_optims(oracle, api, type_, conf)
            g = (rng.standard_normal(sizes[own]) * 1e-2).astype(np.float32)
            assert tables[own].Push(o_gpu, g, 0.01) == 0 and refs[own].push(o_ref, g, 0.01) == 0
            for _ in range(2):
                grads = (rng.standard_normal(grp.n) * 1e-2).astype(np.float32)
                assert grp.CombinePush(o_gpu, grads, 0.01) == 0
                at = 0
                for r, n in zip(refs, sizes):
                    if n:
                        assert r.push(o_ref, grads[at:at + n], 0.01) == 0
                    at += n
            rc, got = grp.CombinePull()
            assert rc == 0
            assert_close(got, np.concatenate([r.pull() for r in refs]), "%d members, %s" % (members, name))
            for t, r, n in zip(tables, refs, sizes):
                for st in STATE_OF[type_] if n else []:
                    ws = r.state(st)
                    assert_close(t.state(st), ws if ws is not None else np.zeros(n, np.float32), "%s state %d" % (name, st))
        grp.close()
        own = members - 2 if members > 1 else 0


@pytest.mark.parametrize("n", [1, 3, 255, 2047, 2048, 2049, 4096, 300_001, (1 << 22) - 1])
@pytest.mark.parametrize("type_", [3, 1])
def test_sparse_pushes_to_small_tables(api, n, type_):
    """Blocking pushes go tile by tile whatever the table's size, and after one whose indices do not ascend by
    fill and scatter for a while: the sequence against a table that takes every gradient dense. Host and device arrays,
    page-locked ones and device memory that is not on 16 bytes too; values are dyadic, so a sum does not depend on its
    order."""
    C, rng = api.C, np.random.default_rng(n)
    w0 = (rng.integers(-64, 65, n) / 64.0).astype(np.float32)
    t, r = api.DenseTable(w0), api.DenseTable(w0)
    opt = api.Optim.create(type_)

    def push(idx, how):
        idx = np.asarray(idx, np.int64)
        val = (rng.integers(-32, 33, idx.size) / 32.0).astype(np.float32)
        inside = (idx >= 0) & (idx < n)
        dense = np.zeros(n, np.float32)
        np.add.at(dense, idx[inside], val[inside])
        if how == "host":
            assert t.PushCoo(opt, idx, val, 0.25) == 0
        elif how == "pinned":
            p = C.c_void_p()
            assert api.lib().krk_host_malloc(C.byref(p), max(1, 12 * idx.size)) == 0
            C.memmove(p, idx.ctypes.data, idx.nbytes)
            C.memmove(p.value + idx.nbytes, val.ctypes.data, val.nbytes)
            assert api.lib().krk_dense_push_coo(t.h, C.byref(opt.raw), p, p.value + idx.nbytes, idx.size, 0.25, 0) == 0
            assert api.lib().krk_host_free(p) == 0
        else:
            skip = int(how == "shifted")
            d_idx = api.DeviceArray.from_host(np.concatenate([np.zeros(skip, np.int64), idx]))
            d_val = api.DeviceArray.from_host(val)
            flags = api.DEVICE_PTRS | (api.ASYNC if how == "async" else 0)
            assert api.lib().krk_dense_push_coo(t.h, C.byref(opt.raw), C.c_void_p(d_idx.ptr + 8 * skip),
                                                C.c_void_p(d_val.ptr), idx.size, 0.25, flags) == 0
            t.sync()
        assert r.Push(opt, dense, 0.25) == 0
        assert np.array_equal(t.Pull()[1], r.Pull()[1]), (idx[:4], how)

    some = np.sort(rng.choice(n, max(1, n // 3), replace=False))
    for how in ("device", "host", "pinned", "shifted", "async"):
        push(some, how)
        push([n - 1], how)
        push(np.arange(n) if n < 5000 else some[:77], how)
    mixed = rng.permutation(np.concatenate([some, some[:1]]))      # an index twice
    for idx in (mixed, np.array([-5, 0]), np.array([n, n + 1]), np.array([0, n])):
        push(idx, "device")
        push(some, "async")
        for _ in range(260 if n in (3, 2049) else 2):               # past the pushes that do not look for tiles
            push(some, "device")
        push(idx, "host")
        push(some, "host")
        push(idx, "pinned")
    push(np.repeat(some, 4)[: n + 2], "device")                    # more entries than elements, where there is room
    t.close()
    r.close()
