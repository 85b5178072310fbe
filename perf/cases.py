"""The work a user has this framework do, as cases that can be timed.

Every case goes through the public entry points: the torch modules of `kraken_amd.torch_embedding`
(a worker's training step), the classes of `kraken_amd.api` (a parameter server's tables, the
gradient codec), and the C entry points of a worker whose server is elsewhere. Ids are hashed
Zipf ranks and gradients are normal, as in `kraken_amd.workloads`; tables hold the rows of the
whole id space before the clock starts, which is the state of a model that has trained for a while,
and one update has been applied, so that the optimizer's state columns exist.

A pass that updates rows ends by reading them again, so that what it returns holds the update.
"""
import functools
import math

import numpy as np
import torch

from kraken_amd import api, dct2
from kraken_amd import torch_embedding as te

OPTIMS = {
    "sgd": (api.OptimType.kSGD, {}, 0),
    "momentum": (api.OptimType.kSGD, {"momentum": "0.9"}, 1),
    "adagrad": (api.OptimType.kAdagrad, {"initial_accumulator": "0.1"}, 1),
    "adam": (api.OptimType.kAdam, {}, 2),
    "rmsprop": (api.OptimType.kRMSprop, {"alpha": "0.9"}, 1),
}
LR = {"sgd": 0.01, "momentum": 0.01, "adagrad": 0.05, "adam": 1e-3, "rmsprop": 1e-3}


# ---------------------------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------------------------
def listed():
    return [
        # one small embedding layer: a request of a hundred ids, where launches and the host count
        dict(name="embedding_small", path="embedding", ids=100, dim=8, rows=100_000, zipf=1.05, optim="sgd"),
        # one field of a click model at an ordinary batch size
        dict(name="embedding_field", path="embedding", ids=8192, dim=64, rows=1_000_000, zipf=1.05, optim="adam"),
        # the duplicate-heavy configuration: a sequence model's ids, wide rows
        dict(name="embedding_dup_heavy", path="embedding", ids=131072 * 8, dim=128, rows=4_000_000, zipf=1.3,
             optim="rmsprop"),
        # Wide&Deep: 26 fields in one combined request, trained through autograd
        dict(name="combine_wide_deep", path="combine", tables=26, batch=8192, dim=16, rows=1_000_000, zipf=1.05,
             optim="adagrad"),
        # the multi-hot fields of the DeepFM configuration, flattened into one jagged batch
        dict(name="jagged_deepfm", path="jagged", bags=65536 * 13, longest=20, dim=32, rows=4_000_000, zipf=1.1,
             optim="adam", mode="mean", weighted=False),
        # 26 multi-hot fields of a smaller batch, a table each
        dict(name="combine_jagged", path="combine_jagged", tables=26, bags=2048, longest=10, dim=16, rows=1_000_000,
             zipf=1.05, optim="adagrad", mode="sum", weighted=False),
        # the server's side of a combined request that is already in GPU memory: unique ids, plus the
        # model's dense parameters (the benchmark's step at dim 32)
        dict(name="server_wide_deep", path="server", tables=26, batch=8192, dim=32, rows=1_000_000, zipf=1.05,
             optim="adagrad", dense=150_000),
        # one RPC's worth of unique ids in the server's own host buffers
        dict(name="host_request", path="host", tables=1, ids=4001, dim=16, rows=200_000, optim="adagrad",
             layout="rows", pinned=False),
        # the dense parameters of one model: pushed and pulled in one combined request
        dict(name="dense_model", path="dense", tables=40, params=434_000, optim="adam"),
        # the gradient codec at its configuration's size: compress, apply to the dense table, pull
        dict(name="codec_full", path="codec", params=4096 * 16384, optim="adam"),
        # the blockwise transform and its inverse at the emitter's default retention
        dict(name="dct2_quarter", path="dct2", blocks=4096 * 64, keep=64),
        # a worker whose server is elsewhere: dedup, expand the reply, sum gradients, route
        dict(name="worker_batch", path="worker", ids=1024 * 26, dim=8, rows=100_000, zipf=1.05),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["embedding", "combine", "jagged", "combine_jagged", "server", "host", "dense", "codec",
                       "dct2", "worker"])
    zipf = rng.choice([1.05, 1.1, 1.3])
    optim = rng.choice(sorted(OPTIMS))
    if path == "embedding":
        return dict(path=path, ids=_log(rng, 64, 1_000_000), dim=rng.choice([8, 10, 16, 32, 48, 64, 100, 128]),
                    rows=_log(rng, 20_000, 4_000_000), zipf=zipf, optim=optim)
    if path == "combine":
        return dict(path=path, tables=rng.randint(2, 32), batch=_log(rng, 32, 12_000), dim=rng.choice([8, 16, 32, 64]),
                    rows=_log(rng, 10_000, 800_000), zipf=zipf, optim=optim)
    if path == "jagged":
        return dict(path=path, bags=_log(rng, 64, 400_000), longest=rng.randint(2, 20), dim=rng.choice([8, 16, 32, 64]),
                    rows=_log(rng, 20_000, 4_000_000), zipf=zipf, optim=optim, mode=rng.choice(["sum", "mean"]),
                    weighted=rng.random() < 0.3)
    if path == "combine_jagged":
        return dict(path=path, tables=rng.randint(2, 26), bags=_log(rng, 32, 4096), longest=rng.randint(2, 15),
                    dim=rng.choice([8, 16, 32]), rows=_log(rng, 10_000, 800_000), zipf=zipf, optim=optim,
                    mode=rng.choice(["sum", "mean"]), weighted=rng.random() < 0.3)
    if path == "server":
        return dict(path=path, tables=rng.randint(1, 32), batch=_log(rng, 32, 16_000), dim=rng.choice([8, 16, 32, 64, 128]),
                    rows=_log(rng, 10_000, 500_000), zipf=zipf, optim=optim, dense=_log(rng, 1000, 1_000_000))
    if path == "host":
        tables = rng.choice([1, 1, 1, rng.randint(2, 26)])
        return dict(path=path, tables=tables, ids=_log(rng, 50, 20_000) // (1 if tables == 1 else 4) + 1,
                    dim=rng.choice([8, 16, 32, 64]), rows=200_000, optim=optim,
                    layout="rows" if tables > 1 else rng.choice(["rows", "wire"]), pinned=rng.random() < 0.5)
    if path == "dense":
        return dict(path=path, tables=rng.choice([1, rng.randint(2, 60)]), params=_log(rng, 5_000, 40_000_000), optim=optim)
    if path == "codec":
        return dict(path=path, params=_log(rng, 300, 60_000_000), optim=optim)
    if path == "dct2":
        return dict(path=path, blocks=_log(rng, 1, 4096 * 50), keep=rng.choice([64, 128, 192, 256]))
    return dict(path=path, ids=_log(rng, 100, 1_500_000), dim=rng.choice([8, 16, 32]), rows=_log(rng, 10_000, 4_000_000),
                zipf=zipf)


# ---------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------
class _Shared:
    """Says where a DeviceArray lies, so that torch can view it."""

    def __init__(self, a):
        kind = "<i8" if a.dtype.kind in "iu" and a.dtype.itemsize == 8 else a.dtype.str
        self.owner = a
        self.__cuda_array_interface__ = dict(shape=a.shape, typestr=kind, data=(a.ptr, False), version=2)


def _array(shape, dtype=np.float32):
    """A zeroed device buffer of the framework and torch's view of it (64-bit ids as int64)."""
    a = api.DeviceArray(shape, dtype)
    return a, torch.as_tensor(_Shared(a), device="cuda").zero_()


def _filled(t):
    """A device buffer of the framework that holds a torch tensor's values; waited for, since the
    framework's objects have streams of their own."""
    a, view = _array(tuple(t.shape), np.uint64 if t.dtype == torch.int64 else np.float32)
    view.copy_(t)
    torch.cuda.synchronize()
    return a


def _int64(c):
    return c - (1 << 64) if c >= 1 << 63 else c


def _hash(x):
    """splitmix64's output function on int64 tensors (the bits of workloads.splitmix64)."""
    def down(v, k):
        return (v >> k) & ((1 << (64 - k)) - 1)
    z = x + _int64(0x9E3779B97F4A7C15)
    z = (z ^ down(z, 30)) * _int64(0xBF58476D1CE4E5B9)
    z = (z ^ down(z, 27)) * _int64(0x94D049BB133111EB)
    return z ^ down(z, 31)


def _table_ids(rows, table=0):
    return _hash(torch.arange(rows, dtype=torch.int64, device="cuda") + table * rows)


@functools.lru_cache(maxsize=4)
def _cdf(zipf, rows):
    c = np.cumsum(np.arange(1, rows + 1, dtype=np.float64) ** -zipf)
    return c / c[-1]


def _zipf_ids(gen, case, n, table=0):
    cdf = torch.from_numpy(_cdf(case["zipf"], case["rows"])).cuda()
    rank = torch.searchsorted(cdf, torch.rand(n, dtype=torch.float64, device="cuda", generator=gen))
    return _hash(rank.clamp_(max=case["rows"] - 1) + table * case["rows"])


def _distinct_ids(gen, case, n, table=0):
    """n distinct Zipf ids in random order: the ids whose exponential arrival times come first."""
    weight = torch.arange(1, case["rows"] + 1, dtype=torch.float64, device="cuda").pow(-case["zipf"])
    arrival = -(1.0 - torch.rand(case["rows"], dtype=torch.float64, device="cuda", generator=gen)).log() / weight
    rank = torch.topk(arrival, n, largest=False).indices.sort().values
    return _hash(rank[torch.randperm(n, device="cuda", generator=gen)] + table * case["rows"])


def _normal(gen, *shape, scale=1e-2):
    return torch.randn(*shape, device="cuda", generator=gen) * scale


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _optim(case):
    kind, conf, _ = OPTIMS[case["optim"]]
    return api.Optim.create(kind, conf)


def _initializer(seed):
    return api.Initializer.create(api.InitializerType.kNormal, {"stddev": "0.01", "seed": str(seed % 1000)})


def _bag_offsets(gen, bags, longest):
    """Bags of 0 to `longest` ids (an empty one yields the patch value)."""
    sizes = torch.randint(0, longest + 1, (bags,), device="cuda", generator=gen)
    sizes[-1] += 1                                       # never an empty batch
    return torch.cat([sizes.new_zeros(1), sizes.cumsum(0)])


def _fill(table, ids, optim, lr):
    """Makes the rows of ids in a SparseTable and applies one (tiny) update."""
    dim = table.dimension
    for part in ids.split(1 << 20):
        assert table.Pull(_filled(part))[0] == 0
    few = _filled(ids[:4])
    grads = _filled(torch.full((min(4, ids.numel()), dim), 1e-3, device="cuda"))
    assert table.Push(optim, few, grads, lr) == 0


# ---------------------------------------------------------------------------------------------
# prepare: what a user's program holds before the call
# ---------------------------------------------------------------------------------------------
def prepare(case, seed):
    return _PREPARE[case["path"]](case, _generator(seed), seed)


def _prepare_embedding(case, gen, seed):
    emb = te.Embedding(case["dim"], initializer=_initializer(seed), optim=_optim(case), lr=LR[case["optim"]],
                       capacity_hint=case["rows"])
    _fill(emb.sparse_table.table(), _table_ids(case["rows"]), _optim(case), LR[case["optim"]])
    return dict(run=_run_module, module=emb, inputs=(_zipf_ids(gen, case, case["ids"]),),
                grads=[_normal(gen, case["ids"], case["dim"])])


def _prepare_combine(case, gen, seed):
    n, dim = case["tables"], case["dim"]
    emb = te.CombineEmbedding([dim] * n, [_initializer(seed + k) for k in range(n)], optim=_optim(case),
                              lr=LR[case["optim"]], capacity_hint=case["rows"])
    for k, t in enumerate(emb.combine_sparse_table.tables()):
        _fill(t, _table_ids(case["rows"], k), _optim(case), LR[case["optim"]])
    # the model lays the fields' rows side by side, so a field's gradient is a block of columns
    return dict(run=_run_module, module=emb, inputs=([_zipf_ids(gen, case, case["batch"], k) for k in range(n)],),
                grads=list(_normal(gen, case["batch"], n * dim).split(dim, dim=1)))


def _jagged_batch(case, gen, table=0):
    offsets = _bag_offsets(gen, case["bags"], case["longest"])
    ids = _zipf_ids(gen, case, int(offsets[-1]), table)
    weights = torch.rand(ids.numel(), device="cuda", generator=gen) + 0.5 if case["weighted"] else None
    return te.JaggedTensor(ids, offsets, weights)


def _prepare_jagged(case, gen, seed):
    emb = te.JaggedEmbedding(case["dim"], initializer=_initializer(seed), optim=_optim(case), lr=LR[case["optim"]],
                             mode=case["mode"], capacity_hint=case["rows"])
    _fill(emb.sparse_table.table(), _table_ids(case["rows"]), _optim(case), LR[case["optim"]])
    return dict(run=_run_module, module=emb, inputs=(_jagged_batch(case, gen),),
                grads=[_normal(gen, case["bags"], case["dim"])])


def _prepare_combine_jagged(case, gen, seed):
    n, dim = case["tables"], case["dim"]
    emb = te.CombineJaggedEmbedding([dim] * n, [_initializer(seed + k) for k in range(n)], modes=[case["mode"]] * n,
                                    optim=_optim(case), lr=LR[case["optim"]], capacity_hint=case["rows"])
    for k, t in enumerate(emb.combine_sparse_table.tables()):
        _fill(t, _table_ids(case["rows"], k), _optim(case), LR[case["optim"]])
    return dict(run=_run_module, module=emb, inputs=([_jagged_batch(case, gen, k) for k in range(n)],),
                grads=list(_normal(gen, case["bags"], n * dim).split(dim, dim=1)))


def _prepare_server(case, gen, seed):
    dim, optim = case["dim"], _optim(case)
    tables = [api.SparseTable(dim, _initializer(seed + k), capacity_hint=case["rows"]) for k in range(case["tables"])]
    for k, t in enumerate(tables):
        _fill(t, _table_ids(case["rows"], k), optim, LR[case["optim"]])
    n = _unique(case, case["batch"])                    # what is left of a batch after the worker's dedup
    parts = [_distinct_ids(gen, case, n, k) for k in range(len(tables))]
    total = sum(p.numel() for p in parts)
    rows, rows_view = _array((total, dim))
    dense = api.DenseTable(_filled(_normal(gen, case["dense"], scale=0.1)))
    params, params_view = _array(case["dense"])
    state = dict(run=_run_server, group=api.TableGroup(tables), optim=optim, lr=LR[case["optim"]],
                 ids=_filled(torch.cat(parts)), offsets=api.TableGroup._offsets([p.numel() for p in parts]),
                 grads=_filled(_normal(gen, total, dim)), rows=rows, rows_view=rows_view,
                 dense=api.DenseGroup([dense]), dense_optim=api.Optim.create(api.OptimType.kAdam),
                 dense_grads=_filled(_normal(gen, case["dense"], scale=1e-3)), params=params, params_view=params_view)
    return state


_ROW_HEADER = [("layout", "u1"), ("rank", "<u8"), ("dim", "<i8"), ("dtype", "u1")]


def _wire_rows(dim):
    """One row of the reference's RPC block: 18 bytes of header, then the values."""
    return np.dtype(_ROW_HEADER + [("vals", "<f4", (dim,))])


def _prepare_host(case, gen, seed):
    dim, optim, n = case["dim"], _optim(case), case["ids"]
    tables = [api.SparseTable(dim, _initializer(seed + k), capacity_hint=case["rows"]) for k in range(case["tables"])]
    parts = []
    for k, t in enumerate(tables):
        every = _table_ids(case["rows"], k)
        _fill(t, every, optim, LR[case["optim"]])
        parts.append(every[torch.randperm(case["rows"], device="cuda", generator=gen)[:n]])
    make = api.pinned_copy if case["pinned"] else np.array
    ids = make(torch.cat(parts).cpu().numpy().view(np.uint64))
    grads = _normal(gen, ids.size, dim).cpu().numpy()
    state = dict(optim=optim, lr=LR[case["optim"]], ids=ids)
    if case["layout"] == "wire":
        block = np.zeros(8 + ids.size * _wire_rows(dim).itemsize, np.uint8)
        block[:8] = np.array([ids.size], np.uint64).view(np.uint8)
        rows = block[8:].view(_wire_rows(dim))
        rows["rank"], rows["dim"], rows["dtype"], rows["vals"] = 1, dim, 11, grads
        # both blocks are 8-byte aligned, as the calls ask
        reply = make(np.zeros(block.size // 8 + 1, np.uint64)).view(np.uint8)[:block.size]
        sent = make(np.zeros(block.size // 8 + 1, np.uint64)).view(np.uint8)[:block.size]
        sent[:] = block
        state.update(run=_run_host_wire, table=tables[0], grads=sent, reply=reply, row=_wire_rows(dim))
    elif len(tables) == 1:
        state.update(run=_run_host_rows, table=tables[0], grads=make(grads), reply=make(np.zeros((ids.size, dim), np.float32)))
    else:
        state.update(run=_run_host_group, group=api.TableGroup(tables), grads=make(grads),
                     offsets=api.TableGroup._offsets([n] * len(tables)), reply=make(np.zeros((ids.size, dim), np.float32)))
    return state


def _dense_sizes(case):
    """A model's parameter tensors: a few large matrices, many small ones, no round sizes."""
    w = np.exp(2.0 * np.random.RandomState(case["tables"]).standard_normal(case["tables"]))
    return [int(s) for s in np.maximum(1, w / w.sum() * case["params"]).astype(np.int64)]


def _prepare_dense(case, gen, seed):
    sizes = _dense_sizes(case)
    tables = [api.DenseTable(_filled(_normal(gen, s, scale=0.1))) for s in sizes]
    params, view = _array(sum(sizes))
    state = dict(run=_run_dense, optim=_optim(case), lr=LR[case["optim"]], group=api.DenseGroup(tables),
                 grads=_filled(_normal(gen, sum(sizes), scale=1e-3)), params=params, view=view)
    return state


def _prepare_codec(case, gen, seed):
    n = case["params"]
    idx, idx_view = _array(n, np.int64)
    val, val_view = _array(n)
    params, params_view = _array(n)
    state = dict(run=_run_codec, bag=api.DenseBag(n), grad=_filled(_normal(gen, n, scale=1.0)), idx=idx, val=val,
                 idx_view=idx_view, val_view=val_view, params=params, params_view=params_view, optim=_optim(case),
                 lr=LR[case["optim"]])
    state["dense"] = api.DenseTable(_filled(_normal(gen, n, scale=0.1)))
    return state


def _prepare_dct2(case, gen, seed):
    n = case["blocks"] * dct2.BLOCK
    coeff, coeff_view = _array((case["blocks"], case["keep"]))
    back, back_view = _array(n)
    state = dict(run=_run_dct2, n=n, keep=case["keep"], x=_filled(_normal(gen, n, scale=1.0)), coeff=coeff,
                 coeff_view=coeff_view, back=back, back_view=back_view)
    return state


def _prepare_worker(case, gen, seed):
    n, dim = case["ids"], case["dim"]
    rng = np.random.default_rng(seed)
    ring_hash = np.sort(rng.integers(0, 1 << 64, 8 * 64, dtype=np.uint64))      # 8 nodes, 64 virtual nodes each
    ids = _zipf_ids(gen, case, n)
    unique = int(torch.unique(ids).numel())
    uids, uids_view = _array(n, np.uint64)
    inv, inv_view = _array(n, np.int64)
    sums, sums_view = _array((n, dim))
    rows, rows_view = _array((n, dim))
    owner, owner_view = _array(n, np.uint64)
    perm, perm_view = _array(n, np.int64)
    state = dict(run=_run_worker, n=n, dim=dim, ring_hash=ring_hash,
                 ring_node=rng.permutation(np.repeat(np.arange(8, dtype=np.uint64), 64)), ids=_filled(ids),
                 grads=_filled(_normal(gen, n, dim)), reply=_filled(_normal(gen, unique, dim)), unique=unique, uids=uids,
                 uids_view=uids_view, inv=inv, inv_view=inv_view, sums=sums, sums_view=sums_view, rows=rows,
                 rows_view=rows_view, owner=owner, owner_view=owner_view, perm=perm, perm_view=perm_view,
                 nodes=np.zeros(8, np.uint64), counts=np.zeros(8, np.int64))
    return state


_PREPARE = dict(embedding=_prepare_embedding, combine=_prepare_combine, jagged=_prepare_jagged,
                combine_jagged=_prepare_combine_jagged, server=_prepare_server, host=_prepare_host,
                dense=_prepare_dense, codec=_prepare_codec, dct2=_prepare_dct2, worker=_prepare_worker)


# ---------------------------------------------------------------------------------------------
# run: one pass
# ---------------------------------------------------------------------------------------------
def run(state):
    return state["run"](state)


def _run_module(s):
    """A training step of the layer (the update is part of backward), then the same batch again
    without gradients, as a program that evaluates after a step reads the rows."""
    out = s["module"](*s["inputs"])
    torch.autograd.backward(out, s["grads"])
    with torch.no_grad():
        after = s["module"](*s["inputs"])
    return out, after


def _run_server(s):
    """A step's pushes, then the pulls of the rows and parameters they changed."""
    s["group"].CombinePush(s["optim"], s["ids"], s["offsets"], s["grads"], s["lr"], async_=True)
    s["dense"].CombinePush(s["dense_optim"], s["dense_grads"], 1e-3, async_=True)
    s["group"].CombinePull(s["ids"], s["offsets"], out=s["rows"], async_=True)
    s["dense"].CombinePull(out=s["params"], async_=True)
    return s["rows_view"], s["params_view"]


def _run_host_rows(s):
    s["table"].Push(s["optim"], s["ids"], s["grads"], s["lr"])
    return s["table"].Pull(s["ids"], out=s["reply"])[1]


def _run_host_wire(s):
    s["table"].PushWire(s["optim"], s["ids"], s["grads"], s["lr"])
    return s["table"].PullWire(s["ids"], reply=s["reply"])[1][8:].view(s["row"])["vals"]


def _run_host_group(s):
    s["group"].CombinePush(s["optim"], s["ids"], s["offsets"], s["grads"], s["lr"])
    return s["group"].CombinePull(s["ids"], s["offsets"], out=s["reply"])[1]


def _run_dense(s):
    s["group"].CombinePush(s["optim"], s["grads"], s["lr"], async_=True)
    s["group"].CombinePull(out=s["params"], async_=True)
    return s["view"]


def _run_codec(s):
    """The worker's compress, the server's apply, the worker's pull."""
    idx, val, nnz = s["bag"].MaybeToCoo(1000, 0.75, s["grad"], idx=s["idx"], val=s["val"])
    api.lib().krk_dense_push_coo(s["dense"].h, api.C.byref(s["optim"].raw), api.C.c_void_p(idx.ptr), api.C.c_void_p(val.ptr),
                                 nnz, s["lr"], api.DEVICE_PTRS)
    s["dense"].Pull(out=s["params"])
    return nnz, s["idx_view"], s["val_view"], s["params_view"]


def _run_dct2(s):
    dct2.forward(s["x"], s["keep"], out=s["coeff"])
    dct2.inverse(s["coeff"], s["n"], s["keep"], out=s["back"])
    return s["coeff_view"], s["back_view"]


def _run_worker(s):
    """Pull side: unique ids, their owners, the reply expanded to the batch. Push side: gradients
    of equal ids summed."""
    lib, p, n, count, nodes = api.lib(), api._ptr, s["n"], api.C.c_int64(), api.C.c_int64()
    lib.krk_dedup(p(s["ids"]), n, p(s["uids"]), p(s["inv"]), api.C.byref(count), api.DEVICE_PTRS)
    u = count.value
    lib.krk_route_ids(7, p(s["ring_hash"]), p(s["ring_node"]), s["ring_hash"].size, p(s["uids"]), u, p(s["owner"]),
                      p(s["perm"]), p(s["nodes"]), p(s["counts"]), 8, api.C.byref(nodes), api.DEVICE_PTRS)
    lib.krk_expand_rows(p(s["reply"]), s["unique"], p(s["inv"]), n, s["dim"], p(s["rows"]), api.DEVICE_PTRS)
    lib.krk_dedup_sum(p(s["ids"]), n, p(s["grads"]), s["dim"], p(s["uids"]), p(s["inv"]), p(s["sums"]),
                      api.C.byref(count), api.DEVICE_PTRS)
    return (u, s["uids_view"], s["inv_view"], s["owner_view"], s["perm_view"], s["nodes"], s["counts"], s["rows_view"],
            s["sums_view"])


# ---------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------
def _unique(case, n):
    """Expected number of distinct ids among n."""
    p = np.diff(_cdf(case["zipf"], case["rows"]), prepend=0.0)
    return max(1, int(round(-np.expm1(n * np.log1p(-np.minimum(p, 0.999999))).sum())))


def _row_bytes(case):
    """A row's key, and its weights and optimizer state read and written."""
    states = OPTIMS[case["optim"]][2]
    return 8 + 8 * case["dim"] * (1 + states) + (16 if case["optim"] == "adam" else 0)


def work(case):
    path = case["path"]
    flops = 0.0
    if path in ("embedding", "combine"):
        tables = case.get("tables", 1)
        n = case.get("ids") or case["batch"]
        # ids and gradients in, the rows of two forwards out, every distinct row updated once
        b = tables * (n * (8 + 12 * case["dim"]) + _unique(case, n) * _row_bytes(case))
    elif path in ("jagged", "combine_jagged"):
        tables = case.get("tables", 1)
        n = case["bags"] * case["longest"] / 2
        b = tables * (n * (12 if case["weighted"] else 8) + case["bags"] * (8 + 12 * case["dim"]) +
                      _unique(case, n) * _row_bytes(case))
    elif path == "server":
        n = case["tables"] * _unique(case, case["batch"])
        b = n * (8 + 8 * case["dim"] + _row_bytes(case)) + case["dense"] * 32
    elif path == "host":
        b = case["tables"] * case["ids"] * (8 + 8 * case["dim"] + _row_bytes(case))
    elif path == "dense":
        b = case["params"] * (4 + 4 + 8 * (1 + OPTIMS[case["optim"]][2]))
    elif path == "codec":
        n, nnz = case["params"], case["params"] / 4
        b = n * (4 + 8) + nnz * 12 + n * 8 * (1 + OPTIMS[case["optim"]][2]) + n * 4
    elif path == "dct2":
        b = 4.0 * case["blocks"] * (2 * 256 + 2 * case["keep"])
        flops = 2.0 * case["blocks"] * 256 * case["keep"]          # folded along the basis' symmetry
    else:
        n, u = case["ids"], _unique(case, case["ids"])
        # ids and gradients in, inv and rows out; uids, owner, perm and sums out, the reply in
        b = n * (8 + 8 + 8 * case["dim"]) + u * (8 * 3 + 8 * case["dim"])
    return {"bytes": float(b), "flops": float(flops)}


def tolerance(case):
    """32-bit sums throughout; indices, inverses and owners are whole numbers and exact. Adam and
    RMSprop divide a summed gradient by its own magnitude, so where the sum cancels to nearly
    nothing a few single elements move by a visible part of one step."""
    if case.get("optim") in ("adam", "rmsprop"):
        return {"rel": 2e-5, "max": 0.2}
    return {"rel": 1e-5, "max": 1e-3}
