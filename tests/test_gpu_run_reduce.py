"""Pushes of up to 2048 and of more than 12288 ids and krk_dedup_sum up to 2^20 ids: pairs grouped by bucket, every bucket
sorted and added up by one workgroup, buckets that hold more pairs than a workgroup takes cut into
chunks and merged. Gradients lie on a binary grid, so that every order of additions gives the same
bits: sums are compared exactly.
"""
import numpy as np
import pytest

from util import splitmix64, zipf_ids

pytestmark = pytest.mark.gpu

MULT = 0x9E3779B1                                       # of the keys' hash


@pytest.fixture(scope="module")
def api():
    from kraken_amd import api as a
    a.lib()
    return a


def _grid(rng, shape):
    return (rng.integers(-64, 65, size=shape) / 4096.0).astype(np.float32)


def _sums(inv, grads, n):
    """Exact while they stay below 2^11."""
    return np.stack([np.bincount(inv, weights=grads[:, c].astype(np.float64), minlength=n) for c in range(grads.shape[1])],
                    1).astype(np.float32)


def _bucket(keys, bits, bucket_bits=10):
    return ((keys.astype(np.uint64) * np.uint64(MULT)) & np.uint64((1 << bits) - 1)) >> np.uint64(bits - bucket_bits)


def _crowded(rng, n, unique, bits, rows):
    """n keys below `unique`, every key once, the others taken in turn from `rows` keys of one bucket: its
    chunks hold more short runs than the merge takes at once."""
    keys = np.arange(unique)
    bucket = _bucket(keys, bits)
    fullest = np.bincount(bucket.astype(np.int64)).argmax()
    crowd = keys[bucket == fullest][:rows]
    assert crowd.size == rows
    return np.concatenate([keys, np.resize(rng.permutation(crowd), n - unique)])


# 128 pairs a bucket: more buckets from 32769 and 65537 pairs on; other tiles from 65537, the counts' scan
# a launch of its own from 262145, longer chunks too; sorted from 2^20 + 1
@pytest.mark.parametrize("n", [1, 8193, 32768, 32769, 65536, 65537, 2**18, 2**18 + 1, 2**20, 2**20 + 1])
@pytest.mark.parametrize("kind", ["distinct", "same", "zipf"])
def test_dedup_sum_sizes(api, n, kind):
    rng = np.random.default_rng(n)
    ids = {"distinct": splitmix64(np.arange(n, dtype=np.uint64)), "same": np.full(n, 7, np.uint64),
           "zipf": zipf_ids(rng, 1.2, 10**5, n)}[kind]
    grads = _grid(rng, (n, 4))
    u, inv, sums = api.dedup_sum(ids, grads)
    assert np.array_equal(u[inv], ids)
    assert np.array_equal(sums, _sums(inv, grads, u.size))


# 2^20 pairs in 1024 buckets: up to 1280 of them are a bucket's one workgroup's, more are cut into chunks of 1024
def test_dedup_sum_whole_and_cut_buckets(api):
    rng = np.random.default_rng(1)
    n, unique = 2**20, 2**19
    keys = np.arange(unique)
    bucket = _bucket(keys, 20).astype(np.int64)
    want = np.full(1024, 1024)
    edges = [1023, 1025, 1279, 1280, 1281, 2047, 2048, 2049]
    want[:len(edges)] = edges
    want[100:340] -= 16                                 # what the edges have more than 1024 each: 3840
    more = [np.resize(keys[bucket == b][:40], want[b] - (bucket == b).sum()) for b in range(1024)]
    keys = np.concatenate([keys, np.concatenate(more)[rng.permutation(n - unique)]])
    grads = _grid(rng, (n, 4))
    u, inv, sums = api.dedup_sum(splitmix64(keys.astype(np.uint64)), grads)
    assert np.array_equal(inv, keys)
    assert np.array_equal(sums, _sums(keys, grads, u.size))


# 39 rows of one bucket 1000 times each: lists of some 5000 entries are sorted in memory; two rows of
# one bucket, the second of which leaves three entries in each of a thousand chunks, more than the
# 2048 that fit at once: window by window. dim 300: a row is more than a wavefront holds
@pytest.mark.parametrize("n", [80_000, 2**20])
@pytest.mark.parametrize("dim", [3, 8, 300])
def test_dedup_sum_crowded_bucket(api, n, dim):
    rng = np.random.default_rng(n + dim)
    if n == 80_000:
        keys = _crowded(rng, n, 40_000, 17, 39)
    else:
        keys = _crowded(rng, n, 2048, 20, 2)
        hot, other = keys[2048], keys[2049]
        keys[2048:] = np.where(np.arange(n - 2048) % 342 == 0, other, hot)
    grads = _grid(rng, (n, dim))
    u, inv, sums = api.dedup_sum(splitmix64(keys.astype(np.uint64)), grads)
    assert np.array_equal(inv, keys)
    assert np.array_equal(sums, _sums(keys, grads, u.size))


# rows whose hash is the same in its upper eight bits: every chunk's list is as long as the chunk, and their
# 13,000 entries, or 4096 with a few to a row's run, are sorted in memory by three digits (2^25 rows of room)
@pytest.mark.parametrize("rows", [2049, 26])
def test_rows_of_one_bucket(api, rows):
    rng = np.random.default_rng(rows)
    t = api.SparseTable(4, api.Initializer.create(api.InitializerType.kConstant, {"value": "1"}))
    t.reserve((1 << 25) - 64)
    names = splitmix64(np.arange(700_000, dtype=np.uint64))
    t.Pull(names)
    bucket = _bucket(t.lookup(names), 25, 8)
    names = names[bucket == np.bincount(bucket.astype(np.int64)).argmax()][:rows]
    assert names.size == rows
    for n in (13_000, 30_000):
        inv = rng.permutation(np.arange(n) % rows)
        grads = _grid(rng, (n, 4))
        before = t.Pull(names)[1]
        assert t.PushRaw(api.Optim.create(api.OptimType.kSGD), names[inv], grads, 0.5) == 0
        assert np.array_equal(t.Pull(names)[1], before - np.float32(0.5) * _sums(inv, grads, rows))


# up to 2048 ids a table every bucket's workgroup picks its pairs out of the request, one to eight a lane; a
# list of up to 256 pairs is sorted by counting
@pytest.mark.parametrize("n", [1, 64, 255, 256, 257, 513, 2047, 2048, 2049])
@pytest.mark.parametrize("dim", [5, 16, 300])
def test_short_requests(api, n, dim):
    rng = np.random.default_rng(n + dim)
    sgd = api.Optim.create(api.OptimType.kSGD)
    tables = [api.SparseTable(dim, api.Initializer.create(api.InitializerType.kConstant, {"value": "1"})) for _ in range(3)]
    group = api.TableGroup(tables[1:])
    for ids in (np.full(n, 3, np.uint64), splitmix64(np.arange(n, dtype=np.uint64)), zipf_ids(rng, 1.3, 5000, n)):
        grads = _grid(rng, (n, dim))
        u, inv = np.unique(ids, return_inverse=True)
        want = np.float32(0.5) * _sums(inv, grads, u.size)
        before = tables[0].Pull(u)[1]
        assert tables[0].PushRaw(sgd, ids, grads, 0.5) == 0
        assert np.array_equal(tables[0].Pull(u)[1], before - want)
        offsets = group._offsets([n // 2, n - n // 2])
        group.CombinePull(ids, offsets)
        before = [t.Pull(u)[1] for t in tables[1:]]
        assert group.CombinePushRaw(sgd, ids, offsets, grads, 0.5) == 0
        for t, b, part in zip(tables[1:], before, (slice(0, n // 2), slice(n // 2, n))):
            assert np.array_equal(t.Pull(u)[1], b - np.float32(0.5) * _sums(inv[part], grads[part], u.size))
        got = api.dedup_sum(ids, grads)
        assert np.array_equal(got[2][np.argsort(got[0])], _sums(inv, grads, u.size))
    group.close()


@pytest.mark.parametrize("dim", [4, 6, 260])
@pytest.mark.parametrize("noted", [False, True])
@pytest.mark.parametrize("shape", ["zipf", "crowded"])
def test_push_raw_and_pooled(api, dim, noted, shape):
    """A table alone, two tables together, bags with weights and means: the same sums."""
    rows, n = 1 << 15, 70_000
    rng = np.random.default_rng(dim + noted)
    names = splitmix64(np.arange(rows, dtype=np.uint64))
    make = lambda: api.SparseTable(dim, api.Initializer.create(api.InitializerType.kConstant, {"value": "1"}),
                                   capacity_hint=1 << 17)
    tables = [make() for _ in range(3)]
    for t in tables:
        t.Pull(names)
    order = np.argsort(tables[0].lookup(names))         # ids by row number
    if shape == "zipf":
        ids = zipf_ids(rng, 1.3, rows, n)
        assert np.isin(ids, names).all()
    else:
        ids = names[order][_crowded(rng, n, rows, 17, 30)]   # 2^17 rows of room
    sgd = api.Optim.create(api.OptimType.kSGD)
    grads = _grid(rng, (n, dim))
    u, inv = np.unique(ids, return_inverse=True)
    d = lambda a: api.DeviceArray.from_host(a)
    d_ids, d_grads, out = d(ids), d(grads), api.DeviceArray((n, dim), np.float32)
    t = tables[0]
    assert t.Pull(d_ids, out=out, note_rows=noted)[0] == 0
    assert t.PushRaw(sgd, d_ids, d_grads, 0.5, as_pulled=noted) == 0
    assert np.array_equal(t.Pull(u)[1], np.float32(1) - np.float32(0.5) * _sums(inv, grads, u.size))
    # together: the second member is the short one
    group = api.TableGroup(tables[1:])
    counts = [n, 500]
    both, g2 = np.concatenate([ids, ids[:500]]), np.concatenate([grads, grads[:500]])
    d_ids, d_grads, out = d(both), d(g2), api.DeviceArray((n + 500, dim), np.float32)
    offsets = group._offsets(counts)
    assert group.CombinePull(d_ids, offsets, out=out, note_rows=noted)[0] == 0
    assert group.CombinePushRaw(sgd, d_ids, offsets, d_grads, 0.5, as_pulled=noted) == 0
    assert np.array_equal(tables[1].Pull(u)[1], np.float32(1) - np.float32(0.5) * _sums(inv, grads, u.size))
    few, back = np.unique(ids[:500], return_inverse=True)
    assert np.array_equal(tables[2].Pull(few)[1], np.float32(1) - np.float32(0.5) * _sums(back, grads[:500], few.size))
    group.close()
    # bags of eight: a mean's ratio is 1/8, weights are powers of two
    bags = n // 8
    bag_grads = _grid(rng, (bags, dim))
    weights = (2.0 ** rng.integers(-1, 2, size=bags * 8)).astype(np.float32)
    for mode, w in (("sum", None), ("mean", None), ("mean", weights)):
        before = t.Pull(u)[1]
        assert t.PushPooled(sgd, ids[:bags * 8], np.arange(bags + 1) * 8, bag_grads, 0.5, mode=mode, weights=w) == 0
        each = np.repeat(bag_grads, 8, 0) * np.float32(1 if mode == "sum" else 0.125)
        if w is not None:
            each = each * w[:, None]
        want = before - np.float32(0.5) * _sums(inv[:bags * 8], each, u.size)
        assert np.array_equal(t.Pull(u)[1], want), mode


@pytest.mark.parametrize("n", [342 * 3072 - 1, 342 * 3072, 342 * 3072 + 1, 2**20 + 1 + 3072])
@pytest.mark.parametrize("unique", [1, 300, 500, 70_000, 2**19 + 3, None])
def test_sorted_requests_by_tiles_and_digits(api, n, unique):
    """Requests that are sorted (more than 2^20 ids): a last tile that is one key short, full, or holds one key, and
    keys of 1, 9, 17, 20 and 21 bits, in one to three passes of seven to nine."""
    rng = np.random.default_rng(n)
    inv = np.arange(n) if unique is None else rng.integers(0, unique, size=n)
    if unique is not None:
        inv[:unique] = np.arange(unique)                # in order of first occurrence
    ids = splitmix64(inv.astype(np.uint64))
    grads = _grid(rng, (n, 1))
    u, got_inv, sums = api.dedup_sum(ids, grads)
    assert np.array_equal(got_inv, inv) and np.array_equal(u, ids[:u.size])
    assert np.array_equal(sums, _sums(inv, grads, u.size))
