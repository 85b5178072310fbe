"""Multi-hot fields: Pull / Push fused with jagged sum / mean pooling, through the C ABI.

The oracle side is the reference's path taken literally: SparseTable::Pull of the ids, the
optional `embeddings *= weights`, then jagged::SumForward / MeanForward
(pytorch/jagged_embedding.py:32-52, pytorch/py/jagged_ops.cc); backwards: Mean/SumBackward,
times the weights, Emitter's dedup + sum, SparseTable::Push. The forward is compared bit for
bit (the GPU adds a bag's rows in the same order); the push like every other push test.
"""
import numpy as np
import pytest

from util import OPTIM_CASES, STATE_OF, assert_close, make_optims, splitmix64

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def api():
    from kraken_amd import api as a
    a.lib()
    return a


def _bags(rng, bags, max_len, space, empty_every=7, pow2=False):
    lengths = rng.integers(1, max_len + 1, size=bags)
    if pow2:
        lengths = 2 ** rng.integers(0, int(np.log2(max_len)) + 1, size=bags)
    lengths[::empty_every] = 0
    off = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)
    ids = splitmix64(rng.integers(0, space, size=int(off[-1])).astype(np.uint64))
    return ids, off


def _tables(api, oracle, dim, seed):
    gi = api.Initializer.create(api.InitializerType.kNormal, {"stddev": "0.01", "seed": str(seed)})
    return api.SparseTable(dim, gi), oracle.SparseTable(dim, oracle.init(oracle.INIT_NORMAL, 0.0, 0.01, seed=seed))


def _oracle_pooled_pull(oracle, ref, ids, off, mode, patch, weights):
    u, inv = oracle.dedup(ids)
    rc, rows = ref.pull(u)
    assert rc == 0
    emb = rows[inv]
    if weights is not None:
        emb = emb * weights[:, None]          # fp32 times fp32, rounded once
    return oracle.jagged_forward(emb, off, mode, patch)


@pytest.mark.parametrize("dim", [8, 16, 32, 128, 6])
@pytest.mark.parametrize("mode", ["sum", "mean"])
@pytest.mark.parametrize("weighted", [False, True])
def test_pooled_pull_matches_pull_then_pool(api, oracle, dim, mode, weighted):
    rng = np.random.default_rng(dim * 7 + weighted)
    t, ref = _tables(api, oracle, dim, seed=dim)
    seen = splitmix64(np.arange(0, 3000, dtype=np.uint64))
    assert t.Pull(seen)[0] == 0 and ref.pull(seen)[0] == 0
    ids, off = _bags(rng, 900, 20, 5000)       # ids 3000..4999 are unseen: inserted by the pull
    w = rng.standard_normal(ids.size).astype(np.float32) if weighted else None
    rc, got = t.PullPooled(ids, off, mode, patch_value=-0.75, weights=w)
    assert rc == 0
    want = _oracle_pooled_pull(oracle, ref, ids, off, mode, -0.75, w)
    assert np.array_equal(got, want)
    assert len(t) == len(ref)
    # the same call again finds every id resident and returns the same bits
    assert np.array_equal(t.PullPooled(ids, off, mode, patch_value=-0.75, weights=w)[1], got)
    # and the inserted rows are the rows a plain Pull returns
    u = np.unique(ids)
    assert np.array_equal(t.Pull(u)[1], ref.pull(u)[1])


def test_pooled_pull_device_arrays_and_edge_shapes(api, oracle):
    rng = np.random.default_rng(3)
    t, ref = _tables(api, oracle, 16, seed=3)
    ids, off = _bags(rng, 4000, 30, 20000)
    d_ids, d_off = api.DeviceArray.from_host(ids), api.DeviceArray.from_host(off)
    rc, d_out = t.PullPooled(d_ids, d_off, "mean", patch_value=2.5)
    assert rc == 0
    assert np.array_equal(d_out.to_host(), _oracle_pooled_pull(oracle, ref, ids, off, "mean", 2.5, None))
    # one bag holding everything, and a field of empty bags only
    one = np.array([0, ids.size], np.int64)
    rc, got = t.PullPooled(ids, one, "sum")
    assert rc == 0 and np.array_equal(got, _oracle_pooled_pull(oracle, ref, ids, one, "sum", 0.0, None))
    rc, got = t.PullPooled(np.zeros(0, np.uint64), np.zeros(6, np.int64), "sum", patch_value=1.25)
    assert rc == 0 and got.shape == (5, 16) and (got == 1.25).all()
    # the same id many times in one bag and across bags
    rep = np.full(1000, ids[0], np.uint64)
    off2 = np.arange(0, 1001, 100, dtype=np.int64)
    rc, got = t.PullPooled(rep, off2, "sum")
    assert rc == 0 and np.array_equal(got, _oracle_pooled_pull(oracle, ref, rep, off2, "sum", 0.0, None))


@pytest.mark.parametrize("dim", [16, 6])
def test_pooled_pulls_while_a_table_is_being_filled(api, oracle, dim):
    """A pooled pull of 8192 positions or more that follows a pull which inserted rows looks its
    positions up without inserting, queues the missing ones and inserts them in a launch of their
    own (rows numbered once per workgroup). Steps whose id space keeps growing (every step brings
    new ids, repeated inside and across bags), then the same request twice: the pooled rows are
    the oracle's bit for bit, and the rows in the table are the rows a plain pull returns."""
    rng = np.random.default_rng(dim)
    t, ref = _tables(api, oracle, dim, seed=40 + dim)
    ids = off = None
    for step in range(6):
        if step < 4:
            ids, off = _bags(rng, 9000, 12, 30_000 * (step + 1))
        assert ids.size >= 32_768
        rc, got = t.PullPooled(ids, off, "mean" if step % 2 else "sum", patch_value=0.5)
        assert rc == 0
        want = _oracle_pooled_pull(oracle, ref, ids, off, "mean" if step % 2 else "sum", 0.5, None)
        assert np.array_equal(got, want), step
        assert len(t) == len(ref)
    u = np.unique(ids)
    assert np.array_equal(t.Pull(u)[1], ref.pull(u)[1])
    gid = t.export()[0]
    assert np.unique(gid).size == gid.size == len(ref)

def test_pooled_argument_errors(api, oracle):
    t, _ = _tables(api, oracle, 16, seed=1)
    ids = np.arange(10, dtype=np.uint64)
    rc, _ = t.PullPooled(ids, np.array([0, 4, 9], np.int64))            # does not end at n
    assert rc == api.E_ARGUMENT
    rc, _ = t.PullPooled(ids, np.array([1, 4, 10], np.int64))           # does not start at 0
    assert rc == api.E_ARGUMENT
    off = np.array([0, 4, 10], np.int64)
    assert t.PullPooled(ids, off)[0] == 0
    _, o_gpu = make_optims(oracle, api, 0, {})
    assert t.PushPooled(o_gpu, ids, off, np.zeros((2, 8), np.float32), 0.1) == api.GRADIENT_UNCOMPATIBLE
    assert t.PushPooled(o_gpu, ids, np.array([0, 4, 9], np.int64), np.zeros((2, 16), np.float32), 0.1) \
        == api.E_ARGUMENT
    other = np.arange(100, 110, dtype=np.uint64)                        # never pulled
    assert t.PushPooled(o_gpu, other, off, np.zeros((2, 16), np.float32), 0.1) == api.SPARSE_ID_NOT_EXIST
    wide, _ = _tables(api, oracle, 512, seed=2)
    assert wide.PullPooled(ids, off)[0] == api.INTERFACE_UNIMPLEMENTED


@pytest.mark.parametrize("case", range(len(OPTIM_CASES)), ids=[c[0] for c in OPTIM_CASES])
@pytest.mark.parametrize("mode,weighted", [("sum", False), ("mean", False), ("mean", True)])
def test_pooled_push_matches_backward_dedup_push(api, oracle, case, mode, weighted):
    _, type_, conf = OPTIM_CASES[case]
    dim = 16
    rng = np.random.default_rng(100 + case)
    t, ref = _tables(api, oracle, dim, seed=case)
    o_ref, o_gpu = make_optims(oracle, api, type_, conf)
    for step in range(3):
        # binary-grid gradients, power-of-two weights and bag lengths: every addend is exact, so
        # the sums do not depend on their order (inexact ratios are covered by
        # test_pooled_push_equals_push_raw_of_the_expanded_gradient)
        ids, off = _bags(rng, 700, 8, 2500, pow2=True)
        bags = off.size - 1
        g = (rng.integers(-64, 65, size=(bags, dim)) / 512.0).astype(np.float32)
        w = (2.0 ** rng.integers(-2, 3, size=ids.size)).astype(np.float32) if weighted else None
        rc, _ = t.PullPooled(ids, off, mode, weights=w)
        assert rc == 0
        ref.pull(oracle.dedup(ids)[0])
        assert t.PushPooled(o_gpu, ids, off, g, 0.05, mode=mode, weights=w) == 0
        vg = oracle.jagged_backward(off, g, mode)
        if w is not None:
            vg = vg * w[:, None]
        u, gs = oracle.dedup_sum(ids, vg)
        assert ref.push(o_ref, u, gs, 0.05) == 0
    for st in STATE_OF[type_]:
        rid, rval, rstate, rsteps = ref.export(state_type=st)
        gid, gval, gstate, gsteps = t.export(state_type=st)
        a, b = np.argsort(rid), np.argsort(gid)
        assert np.array_equal(rid[a], gid[b])
        assert_close(gval[b], rval[a], "weights")
        if rstate is not None and gstate is not None:
            assert_close(gstate[b], rstate[a], "state %d" % st)
        if type_ == 1:
            assert np.array_equal(gsteps[b], rsteps[a])


def test_pooled_push_equals_push_raw_of_the_expanded_gradient(api, oracle):
    """Size-independent property: the pooled push is PushRaw of the per-position gradient the
    worker would have materialised (inexact mean ratios and arbitrary weights included). Two
    tables number their rows differently, so the additions are grouped differently: SGD keeps
    the comparison well conditioned (the update is linear in the summed gradient), and the
    tolerance is that of two fp32 summation orders, far below one wrong ratio or weight."""
    dim, n_bags = 32, 60000
    rng = np.random.default_rng(8)
    ids, off = _bags(rng, n_bags, 20, 200000)
    g = (rng.standard_normal((n_bags, dim)) * 1e-2).astype(np.float32)
    w = rng.standard_normal(ids.size).astype(np.float32)
    u = np.unique(ids)
    for mode, weights in (("sum", None), ("mean", None), ("sum", w), ("mean", w)):
        a, _ = _tables(api, oracle, dim, seed=5)
        b, _ = _tables(api, oracle, dim, seed=5)
        assert a.Pull(u)[0] == 0 and b.Pull(u)[0] == 0
        before = a.Pull(u)[1]
        _, o_gpu = make_optims(oracle, api, 3, {})
        for _ in range(2):
            assert a.PushPooled(o_gpu, ids, off, g, 0.5, mode=mode, weights=weights) == 0
            vg = oracle.jagged_backward(off, g, mode)
            if weights is not None:
                vg = vg * weights[:, None]
            assert b.PushRaw(o_gpu, ids, vg, 0.5) == 0
        wa, wb = a.Pull(u)[1], b.Pull(u)[1]
        moved = np.abs(wb - before).max()
        assert moved > 1e-3                                   # the pushes did something
        assert np.abs(wa - wb).max() <= 1e-6 * max(1.0, moved * 10), (mode, weights is not None)


@pytest.mark.parametrize("bags", [[300, 0, 1, 700], [6000, 20, 0, 700]], ids=["short", "long"])
@pytest.mark.parametrize("dim", [16, 6])
@pytest.mark.parametrize("noted", [False, True])
def test_combined_pooled_pull_and_push(api, oracle, bags, dim, noted):
    """krk_group_pull_pooled_parts / krk_group_push_pooled_parts over members that differ in mode and
    weights, one of them empty, one with positions outside every bag, gradients that are columns of
    a wider matrix; requests on both sides of the 12288 ids a member up to which a push is two
    launches, new ids every step, with and without the row notes of the pull. Binary-grid values:
    every sum is exact, so the rows are the oracle's bit for bit."""
    C = api.C

    class Part(C.Structure):
        _fields_ = [("ids", C.c_void_p), ("n", C.c_int64), ("offsets", C.c_void_p), ("bags", C.c_int64),
                    ("weights", C.c_void_p), ("rows", C.c_void_p), ("stride", C.c_int64), ("mode", C.c_int32),
                    ("patch", C.c_float)]

    rng = np.random.default_rng(dim + len(bags) + noted)
    modes, weighted = ["sum", "mean", "sum", "mean"], [False, False, True, True]
    pairs = [_tables(api, oracle, dim, seed=70 + k) for k in range(4)]
    group = api.TableGroup([t for t, _ in pairs])
    o_ref, o_gpu = make_optims(oracle, api, 3, {})
    flags = api.DEVICE_PTRS
    for step in range(3):
        parts, push, host, keep = (Part * 4)(), (Part * 4)(), [], []
        wide = (rng.integers(-64, 65, size=(max(bags), 4, dim)) / 512.0).astype(np.float32)
        d_wide = api.DeviceArray.from_host(wide.reshape(max(bags), 4 * dim))
        for k in range(4):
            ids, off = _bags(rng, bags[k], 8, 1500 * (step + 1), pow2=True) if bags[k] else (
                np.zeros(0, np.uint64), np.zeros(1, np.int64))
            if k == 3:                                     # two positions ahead of the bags, one behind
                ids = np.concatenate([ids[:1], ids[-1:], ids, ids[:1]]) + np.uint64(1)
                off = off + 2
            w = (2.0 ** rng.integers(-2, 3, size=ids.size)).astype(np.float32) if weighted[k] else None
            d = [api.DeviceArray.from_host(a) if a is not None and a.size else None for a in (ids, off, w)]
            out = api.DeviceArray((max(bags[k], 1), dim), np.float32)
            keep.append((d, out))
            ptr = [x.ptr if x is not None else None for x in d]
            mode = 0 if modes[k] == "sum" else 1
            parts[k] = Part(ptr[0], ids.size, ptr[1], bags[k], ptr[2], out.ptr, dim, mode, 0.25)
            push[k] = Part(ptr[0], ids.size, ptr[1], bags[k], ptr[2], d_wide.ptr + 4 * dim * k, 4 * dim, mode, 0.0)
            host.append((ids, off, w, out))
        api._check(api.lib().krk_group_pull_pooled_parts(group.h, parts, flags | (api.NOTE_ROWS if noted else 0)), "pull")
        for k, (ids, off, w, out) in enumerate(host):
            if not bags[k]:
                continue
            ref = pairs[k][1]
            ref.pull(oracle.dedup(ids)[0])                 # rows are made in the order the oracle meets them
            lo, hi = int(off[0]), int(off[-1])
            want = _oracle_pooled_pull(oracle, ref, ids[lo:hi], off - lo, modes[k], 0.25, w[lo:hi] if w is not None else None)
            assert np.array_equal(out.to_host(), want), (step, k)
        api._check(api.lib().krk_group_push_pooled_parts(group.h, C.byref(o_gpu.raw), push, dim, 0.5,
                                                         flags | (api.IDS_AS_PULLED if noted else 0)), "push")
        for k, (ids, off, w, _) in enumerate(host):
            if not bags[k]:
                continue
            lo, hi = int(off[0]), int(off[-1])
            vg = oracle.jagged_backward(off - lo, np.ascontiguousarray(wide[:bags[k], k]), modes[k])
            if w is not None:
                vg = vg * w[lo:hi, None]
            u, gs = oracle.dedup_sum(ids[lo:hi], vg)
            assert pairs[k][1].push(o_ref, u, gs, 0.5) == 0
            every = np.unique(ids)
            assert np.array_equal(pairs[k][0].Pull(every)[1], pairs[k][1].pull(every)[1]), (step, k)
            assert len(pairs[k][0]) == len(pairs[k][1])
    missing = splitmix64(np.arange(10**7, 10**7 + 40, dtype=np.uint64))
    d_ids, d_off = api.DeviceArray.from_host(missing), api.DeviceArray.from_host(np.array([0, 40], np.int64))
    one = (Part * 4)()
    one[0] = Part(d_ids.ptr, 40, d_off.ptr, 1, None, keep[0][1].ptr, dim, 0, 0.0)
    assert api.lib().krk_group_push_pooled_parts(group.h, C.byref(o_gpu.raw), one, dim, 0.5, flags) == api.SPARSE_ID_NOT_EXIST
    group.close()


@pytest.mark.parametrize("filler", [0, 14_000], ids=["short", "long"])
@pytest.mark.parametrize("noted", [False, True])
@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("grouped", [False, True])
def test_offsets_that_descend_stay_inside_the_request(api, filler, noted, weighted, grouped):
    """Offsets on the device are not read back to be checked. Where they descend, a position between the
    first and the last offset belongs to a bag that the offsets step over it with, every other position to
    none, whatever bags reach over it; nothing outside the arrays is read. Bags that overlap have the
    same gradient row here, so that it does not matter which of them a position is given to."""
    C, dim, n = api.C, 4, 40 + filler
    gi = api.Initializer.create(api.InitializerType.kConstant, {"value": "1"})
    t = api.SparseTable(dim, gi)
    group = api.TableGroup([t]) if grouped else None
    sgd = api.Optim.create(api.OptimType.kSGD)
    ids = splitmix64(np.arange(n, dtype=np.uint64))
    d_ids = api.DeviceArray.from_host(ids)
    w = np.full(n, 0.5, np.float32) if weighted else None
    d_w = api.DeviceArray.from_host(w) if weighted else None
    p = lambda x: C.c_void_p(x.ptr) if x is not None else None
    top = n - 10
    for off in ([5, 2, 8, 8, 20, 11, top], [top, 30, 5], [0, n + 7, -3, n], [-(1 << 40), 7, 1 << 40], [12, 12, 12],
                [n + 100, 3, 9, n + 200], [3, -1, -9]):
        off = np.array(off, np.int64)
        bags = off.size - 1
        d_off = api.DeviceArray.from_host(off)
        d_g = api.DeviceArray.from_host(np.ones((bags, dim), np.float32))
        out = api.DeviceArray((bags, dim), np.float32)
        before = t.Pull(ids)[1]
        flags = api.DEVICE_PTRS
        note, pulled = (api.NOTE_ROWS, api.IDS_AS_PULLED) if noted else (0, 0)
        if grouped:
            class Part(C.Structure):
                _fields_ = [("ids", C.c_void_p), ("n", C.c_int64), ("offsets", C.c_void_p), ("bags", C.c_int64),
                            ("weights", C.c_void_p), ("rows", C.c_void_p), ("stride", C.c_int64), ("mode", C.c_int32),
                            ("patch", C.c_float)]
            part = lambda rows: (Part * 1)(Part(d_ids.ptr, n, d_off.ptr, bags, d_w.ptr if weighted else None, rows.ptr,
                                                dim, 0, 0.0))
            assert api.lib().krk_group_pull_pooled_parts(group.h, part(out), flags | note) == 0
            assert api.lib().krk_group_push_pooled_parts(group.h, C.byref(sgd.raw), part(d_g), dim, 0.5,
                                                         flags | pulled) == 0
        else:
            assert api.lib().krk_sparse_pull_pooled(t.h, p(d_ids), n, p(d_off), bags, p(d_w), 0, 0.0, p(out),
                                                    flags | note) == 0
            assert api.lib().krk_sparse_push_pooled(t.h, C.byref(sgd.raw), p(d_ids), n, p(d_off), bags, p(d_w), 0,
                                                    p(d_g), dim, 0.5, flags | pulled) == 0
        at = np.arange(n)
        moved = (at >= off[0]) & (at < off[-1])
        want = before - np.float32(0.25 if weighted else 0.5) * moved[:, None].astype(np.float32)
        assert np.array_equal(t.Pull(ids)[1], want), off[:3]
    if group:
        group.close()


# a wavefront looks 64 ids up together; the last of the table's buckets are chained where it is half full
@pytest.mark.parametrize("n", [1, 15, 16, 63, 64, 65, 255, 257, 5000])
@pytest.mark.parametrize("dim", [4, 6, 32])
def test_pooled_pulls_find_every_id(api, n, dim):
    """Resident ids, ids that are made by the call, repeats of both, and the id that equals the index's
    empty marker, in one pull; the rows against a plain pull's, added in position order."""
    rng = np.random.default_rng(n + dim)
    t = api.SparseTable(dim, api.Initializer.create(api.InitializerType.kNormal, {"stddev": "1", "seed": "5"}),
                        capacity_hint=4096)
    t.Pull(splitmix64(np.arange(3500, dtype=np.uint64)))
    ids = splitmix64(rng.integers(0, 4000, n).astype(np.uint64))
    ids[rng.integers(0, n, max(1, n // 20))] = np.uint64(2**64 - 1)
    cuts = np.sort(rng.integers(0, n + 1, max(1, n // 4)))
    offsets = np.concatenate([[0], cuts, [n]]).astype(np.int64)
    rc, got = t.PullPooled(ids, offsets)
    assert rc == 0
    rows = t.Pull(ids)[1]
    want = np.zeros((offsets.size - 1, dim), np.float32)
    for b in range(offsets.size - 1):
        for j in range(offsets[b], offsets[b + 1]):
            want[b] = rows[j] if j == offsets[b] else want[b] + rows[j]
    assert np.array_equal(got, want)
    assert len(t) == np.union1d(ids, splitmix64(np.arange(3500, dtype=np.uint64))).size


# A pull below 8192 ids takes sixteen ids a wavefront while many are new, and for eight pulls after, 64
# otherwise, whose missing ids are moved together sixteen at a time; from 8192 on new ids are queued.
@pytest.mark.parametrize("n", [17, 64, 65, 1000, 8191, 8192])
@pytest.mark.parametrize("dim", [6, 32])
@pytest.mark.parametrize("combined", [False, True])
def test_pooled_pulls_make_rows(api, n, dim, combined):
    """Pulls with no, few and only new ids in turn, more than eight with none between them; bags of one
    id, so that a bag is its row: against a plain pull of the same ids."""
    C = api.C

    class Part(C.Structure):
        _fields_ = [("ids", C.c_void_p), ("n", C.c_int64), ("offsets", C.c_void_p), ("bags", C.c_int64),
                    ("weights", C.c_void_p), ("rows", C.c_void_p), ("stride", C.c_int64), ("mode", C.c_int32),
                    ("patch", C.c_float)]

    rng = np.random.default_rng(n + dim)
    gi = api.Initializer.create(api.InitializerType.kNormal, {"stddev": "1", "seed": "5"})
    tables = [api.SparseTable(dim, gi, capacity_hint=64) for _ in range(2 if combined else 1)]
    group = api.TableGroup(tables) if combined else None
    offsets = api.DeviceArray.from_host(np.arange(n + 1, dtype=np.int64))
    made = 0
    for step, share in enumerate([1.0, 0.3, 0.0, 1.0] + [0.0] * 10 + [0.02, 0.3, 1.0, 0.02]):
        fresh = np.arange(made, made + int(np.ceil(n * share)), dtype=np.uint64)
        made += fresh.size
        ids, outs = [], []
        for _ in tables:
            old = rng.integers(0, made, n - fresh.size).astype(np.uint64)
            ids.append(splitmix64(np.concatenate([fresh, old])[rng.permutation(n)]))
            outs.append(api.DeviceArray((n, dim), np.float32))
        d_ids = [api.DeviceArray.from_host(i) for i in ids]
        if group:
            parts = (Part * 2)(*[Part(d.ptr, n, offsets.ptr, n, None, o.ptr, dim, 0, 0.0) for d, o in zip(d_ids, outs)])
            assert api.lib().krk_group_pull_pooled_parts(group.h, parts, api.DEVICE_PTRS) == 0
        else:
            assert tables[0].PullPooled(d_ids[0], offsets, out=outs[0])[0] == 0
        for t, i, o in zip(tables, ids, outs):
            assert len(t) == made, (step, len(t))
            assert np.array_equal(o.to_host(), t.Pull(i)[1]), step
    if group:
        group.close()


@pytest.mark.parametrize("dim,groups", [(8, 32), (32, 8), (128, 2), (10, 4)])
@pytest.mark.parametrize("per_wavefront", [1, 2, 32])
def test_pooled_pulls_of_many_bags(api, dim, groups, per_wavefront):
    """Requests from whose number of bags on a wavefront takes more of them than it has lane groups (twice and up
    to 64 as many), with a last wavefront that is not full; sums in position order, bit for bit."""
    bags = min(8192 * groups * per_wavefront, 8192 * 64) + 5
    rng = np.random.default_rng(dim + per_wavefront)
    t = api.SparseTable(dim, api.Initializer.create(api.InitializerType.kNormal, {"stddev": "0.01", "seed": "4"}))
    every = splitmix64(np.arange(500, dtype=np.uint64))
    rc, rows = t.Pull(every)
    assert rc == 0
    lengths = rng.choice([0, 1, 2, 4, 5, 9], size=bags, p=[.3, .3, .2, .1, .05, .05])
    off = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)
    pick = rng.integers(0, every.size, size=int(off[-1]))
    w = rng.standard_normal(pick.size).astype(np.float32)
    want = np.full((bags, dim), -0.75, np.float32)
    weighted = want.copy()
    for u in range(int(lengths.max())):
        on = np.flatnonzero(lengths > u)
        at = off[:-1][on] + u
        row = rows[pick[at]]
        want[on] = row if u == 0 else want[on] + row
        row = row * w[at][:, None]
        weighted[on] = row if u == 0 else weighted[on] + row
    d_ids, d_off = api.DeviceArray.from_host(every[pick]), api.DeviceArray.from_host(off)
    rc, got = t.PullPooled(d_ids, d_off, "sum", patch_value=-0.75)
    assert rc == 0 and np.array_equal(got.to_host(), want)
    rc, got = t.PullPooled(d_ids, d_off, "mean", patch_value=-0.75, weights=api.DeviceArray.from_host(w))
    some = lengths > 0
    weighted[some] *= (1.0 / lengths[some]).astype(np.float32)[:, None]
    assert rc == 0 and np.array_equal(got.to_host(), weighted)


def _in_order(rows, off, w, mean, patch):
    """The bags' sums in position order, in fp32: rows are the positions' (jagged_ops.cc:205-224)."""
    lengths = np.diff(off)
    want = np.full((lengths.size, rows.shape[1]), patch, np.float32)
    for u in range(int(lengths.max(initial=0))):
        on = np.flatnonzero(lengths > u)
        row = rows[off[:-1][on] + u]
        if w is not None:
            row = row * w[off[:-1][on] + u][:, None]
        want[on] = row if u == 0 else want[on] + row
    if mean:
        some = lengths > 0
        want[some] *= (1.0 / lengths[some]).astype(np.float32)[:, None]
    return want


# Rows of 128 floats: a wavefront has two lane groups, and takes 4 bags from 32,768 on, 64 from 524,288 on. Of 32 floats
# eight groups and 16 bags from 131,072 on, of 8 floats 32 and 64 from 524,288 on, of 10 floats four and 8 from 65,536 on.
@pytest.mark.parametrize("dim,bags", [(128, (32_768,)), (128, (40_000, 0, 7)), (128, (12_000, 11_500, 12_001)),
                                      (128, (32_766, 1, 1)), (128, (6, 524_300)), (32, (140_000, 3)), (32, (524_289,)),
                                      (8, (524_290,)), (8, (300_000, 299_000)), (10, (70_000, 9))])
def test_combined_pooled_pulls_of_many_bags(api, dim, bags):
    """Members of which a wavefront takes more bags than it has lane groups: one, unequal ones (of no bag, of fewer than
    a wavefront takes), equal ones, with two stretches of long bags that are shared out among wavefronts; ids that
    the request itself makes, each at many positions, so that positions read an id's row while another one is
    making it; then the same request over rows that are there, and the first member's part by itself."""
    C = api.C

    class Part(C.Structure):
        _fields_ = [("ids", C.c_void_p), ("n", C.c_int64), ("offsets", C.c_void_p), ("bags", C.c_int64),
                    ("weights", C.c_void_p), ("rows", C.c_void_p), ("stride", C.c_int64), ("mode", C.c_int32),
                    ("patch", C.c_float)]

    rng = np.random.default_rng(sum(bags))
    gi = api.Initializer.create(api.InitializerType.kNormal, {"stddev": "0.01", "seed": "4"})
    tables = [api.SparseTable(dim, gi, capacity_hint=64) for _ in bags]
    group = api.TableGroup(tables)
    made, held = [], []
    for m, count in enumerate(bags):
        lengths = rng.choice([0, 1, 2, 4, 5], size=count, p=[.3, .4, .2, .05, .05])
        lengths[1001:1300] = 40
        lengths[-101:] = rng.integers(20, 40, lengths[-101:].size)
        off = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)
        ids = splitmix64(rng.integers(0, 60, size=int(off[-1])).astype(np.uint64))
        ids[::97] = np.uint64(2**64 - 1)
        w = rng.standard_normal(ids.size).astype(np.float32) if m % 2 == 0 else None
        out = api.DeviceArray((max(count, 1), dim), np.float32)
        d_ids, d_off = api.DeviceArray.from_host(ids), api.DeviceArray.from_host(off)
        d_w = api.DeviceArray.from_host(w) if w is not None else None
        held.append((d_ids, d_off, d_w))
        made.append((ids, off, w, m % 3 == 1, -0.75 - m, out))
    parts = (Part * len(bags))(*[Part(h[0].ptr, i.size, h[1].ptr, off.size - 1, h[2].ptr if h[2] else None, out.ptr, dim,
                                      1 if mean else 0, patch)
                                 for h, (i, off, w, mean, patch, out) in zip(held, made)])
    for step in range(2):
        assert api.lib().krk_group_pull_pooled_parts(group.h, parts, api.DEVICE_PTRS) == 0
        for t, (ids, off, w, mean, patch, out) in zip(tables, made):
            if off.size == 1:
                continue
            u, inv = np.unique(ids, return_inverse=True)
            rows = t.Pull(u)[1][inv] if u.size else np.zeros((0, dim), np.float32)
            assert len(t) == u.size
            want = _in_order(rows, off, w, mean, patch)
            assert np.array_equal(out.to_host(), want), step
            if t is tables[0]:
                rc, got = t.PullPooled(held[0][0], held[0][1], "mean" if mean else "sum", patch_value=patch, weights=held[0][2])
                assert rc == 0 and np.array_equal(got.to_host(), want), step
    group.close()


def test_pooled_pulls_of_uneven_bags_take_no_longer_in_order(api):
    """Long bags that stand together (bags in order of their length, one field's histories behind the other fields'
    single ids) are shared out among wavefronts. As 64 neighbours of one wavefront this request took seven
    times as long in order as shuffled; it is to take no more than twice as long."""
    rng = np.random.default_rng(3)
    dim, bags, rows = 32, 8192 * 64 + 5, 100_000
    t = api.SparseTable(dim, api.Initializer.create(api.InitializerType.kConstant, {"value": "1"}), rows)
    every = splitmix64(np.arange(rows, dtype=np.uint64))
    assert t.Pull(every)[0] == 0
    lengths = np.minimum(3000, np.floor(3.5 * rng.pareto(1.3, bags))).astype(np.int64)
    d_ids = api.DeviceArray.from_host(every[rng.integers(0, rows, size=int(lengths.sum()))])
    out = api.DeviceArray((bags, dim), np.float32)
    took = {}
    for order, per_bag in (("shuffled", lengths), ("ascending", np.sort(lengths)), ("descending", np.sort(lengths)[::-1])):
        d_off = api.DeviceArray.from_host(np.concatenate([[0], np.cumsum(per_bag)]).astype(np.int64))
        begin, end = api.Event(), api.Event()
        each = []
        for _ in range(5):
            begin.record(t)
            assert t.PullPooled(d_ids, d_off, out=out, async_=True)[0] == 0
            end.record(t)
            t.sync()
            each.append(begin.elapsed_ms(end))
        took[order] = min(each)
        assert np.array_equal(out.to_host()[:, 0], per_bag.astype(np.float32)), order
    assert max(took["ascending"], took["descending"]) <= 2 * took["shuffled"], took
