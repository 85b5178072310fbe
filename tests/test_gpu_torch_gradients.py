"""The gradients that autograd hands to the embedding modules in all the forms it has: none at all,
zeros that were never made, blocks of a wider matrix that start anywhere, one value expanded over
the batch. Whatever the form, the tables end as the oracle's, pushed with the same gradients in plain
arrays (an output without a gradient pushes zeros, pytorch/combine_embedding.py:22-31)."""
import gc

import numpy as np
import pytest

from util import assert_close, make_optims

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

KINDS = ["embedding", "jagged", "combine", "combine_jagged"]
DIM = 16
LR = 0.5


@pytest.fixture(scope="module")
def mods():
    if not torch.cuda.is_available():
        pytest.skip("torch sees no GPU")
    from kraken_amd import api, torch_embedding
    api.lib()
    return api, torch_embedding


class Pair:
    """A module of `kind` over the oracle's tables with the same rows and optimizer."""

    def __init__(self, mods, oracle, kind, optim=(1, {}), seed=40):
        self.api, self.te = mods
        self.oracle, self.kind = oracle, kind
        self.jagged = "jagged" in kind
        self.tables = 2 if kind.startswith("combine") else 1
        api, te = mods
        inits = [api.Initializer.create(api.InitializerType.kNormal, {"stddev": "0.01", "seed": str(seed + i)})
                 for i in range(self.tables)]
        self.refs = [oracle.SparseTable(DIM, oracle.init(oracle.INIT_NORMAL, 0.0, 0.01, seed=seed + i))
                     for i in range(self.tables)]
        self.o_ref, self.o_gpu = make_optims(oracle, api, *optim)
        if kind == "embedding":
            self.mod = te.Embedding(DIM, inits[0], self.o_gpu, LR)
        elif kind == "jagged":
            self.mod = te.JaggedEmbedding(DIM, inits[0], self.o_gpu, LR, mode="sum")
        elif kind == "combine":
            self.mod = te.CombineEmbedding([DIM] * 2, inits, self.o_gpu, LR)
        else:
            self.mod = te.CombineJaggedEmbedding([DIM] * 2, inits, ["sum", "mean"], None, self.o_gpu, LR)
        self.param = self.mod.sparse_table if self.tables == 1 else self.mod.combine_sparse_table
        self.held = [self.param.table()] if self.tables == 1 else self.param.tables()
        self.modes = ["sum", "mean"]

    def draw(self, rng, rows, span=200):
        """-> per table (ids, offsets or None): `rows` output rows each"""
        batch = []
        for _ in range(self.tables):
            if self.jagged:
                off = np.concatenate([[0], np.cumsum(rng.choice([1, 2, 4], size=rows))]).astype(np.int64)
                batch.append((rng.integers(0, span, size=int(off[-1])).astype(np.uint64), off))
            else:
                batch.append((rng.integers(0, span, size=rows).astype(np.uint64), None))
        return batch

    def tensors(self, batch):
        return [(torch.from_numpy(ids.astype(np.int64)).cuda(), None if off is None else torch.from_numpy(off).cuda())
                for ids, off in batch]

    def forward(self, batch, tensors=None):
        """-> the module's outputs as a list, checked against the oracle's rows"""
        t = tensors or self.tensors(batch)
        if self.kind == "embedding":
            outs = [self.mod(t[0][0])]
        elif self.kind == "jagged":
            outs = [self.mod(*t[0])]
        elif self.kind == "combine":
            outs = self.mod([ids for ids, _ in t])
        else:
            outs = self.mod([self.te.JaggedTensor(ids, off) for ids, off in t])
        for i, (ids, off) in enumerate(batch):
            u, inv = self.oracle.dedup(ids)
            rows = self.refs[i].pull(u)[1][inv]
            want = rows if off is None else self.oracle.jagged_forward(rows, off, self.modes[i], 0.0)
            assert_close(outs[i].detach().cpu().numpy(), want, "forward of table %d" % i, rtol=1e-5, atol=1e-6)
        return outs

    def push(self, batch, grads):
        """the oracle's update; grads: an array per table, [its output rows, DIM]"""
        for i, ((ids, off), g) in enumerate(zip(batch, grads)):
            vg = g if off is None else self.oracle.jagged_backward(off, g, self.modes[i])
            u, sums = self.oracle.dedup_sum(ids, vg)
            assert self.refs[i].push(self.o_ref, u, sums, LR) == 0

    def check(self, what):
        torch.cuda.synchronize()
        for i, (t, r) in enumerate(zip(self.held, self.refs)):
            rid, rval, _, _ = r.export()
            assert len(t) == len(r)
            assert_close(t.Pull(rid)[1], rval, "%s: rows of table %d" % (what, i), rtol=1e-5, atol=1e-6)


def _coef(rng, rows, n):
    return [(rng.integers(-8, 9, size=(rows, DIM)) / 16.0).astype(np.float32) for _ in range(n)]


def _loss(outs, coefs):
    return sum((o * torch.from_numpy(c).cuda()).sum() for o, c in zip(outs, coefs) if c is not None)


# optimizers for which a gradient of zeros still moves the row, its state or its counter
MOVING = [("adam", 1, {}), ("momentum", 3, {"momentum": 0.9}), ("sgd_decay", 3, {"weight_decay": 0.05}),
          ("rmsprop", 2, {"momentum": 0.7})]


@pytest.mark.parametrize("optim", MOVING, ids=[m[0] for m in MOVING])
@pytest.mark.parametrize("kind", ["combine", "combine_jagged"])
def test_output_without_gradient_pushes_zeros(mods, oracle, kind, optim):
    """A loss that uses one of two outputs: the rows of the other take their step with zeros."""
    p = Pair(mods, oracle, kind, optim[1:])
    rng = np.random.default_rng(1)
    for step in range(3):
        batch = p.draw(rng, 96)
        outs = p.forward(batch)
        coefs = _coef(rng, 96, 2)
        used = [coefs[0], None if step == 1 else coefs[1]]
        _loss(outs, used).backward()
        p.push(batch, [np.zeros_like(c) if u is None else c for c, u in zip(coefs, used)])
    p.check("after a step without the second output")


@pytest.mark.parametrize("kind", KINDS)
def test_a_closed_table_is_refused(mods, oracle, kind):
    """After close() a forward, and the backward of an earlier forward (in autograd's thread), raise."""
    p = Pair(mods, oracle, kind)
    rng = np.random.default_rng(7)
    batch = p.draw(rng, 32)
    outs = p.forward(batch)
    if kind == "combine":
        for group in p.param._groups.values():
            group.close()
    p.held[-1].close()                           # of a pooled request, one table is enough
    gc.collect()
    with pytest.raises(p.api.KrakenHipError):
        _loss(outs, _coef(rng, 32, p.tables)).backward()
    with pytest.raises(p.api.KrakenHipError):
        p.forward(batch)


@pytest.mark.parametrize("kind", KINDS)
def test_another_optimizer_between_forward_and_backward(mods, oracle, kind):
    """The optimizer that a table has when backward runs is the one that counts, replaced or changed."""
    p = Pair(mods, oracle, kind, (3, {}))
    rng = np.random.default_rng(8)
    for step in range(3):
        batch = p.draw(rng, 48)
        outs = p.forward(batch)
        if step == 1:
            p.o_ref, p.param._optim = make_optims(oracle, p.api, 0, {"eps": 1e-6})
            p.o_gpu = None
            gc.collect()
        elif step == 2:
            p.o_ref, _ = make_optims(oracle, p.api, 0, {"eps": 0.125})
            p.param._optim.raw.eps = 0.125
        coefs = _coef(rng, 48, p.tables)
        _loss(outs, coefs).backward()
        p.push(batch, coefs)
    p.check("after changes of the optimizer")


@pytest.mark.parametrize("kind", KINDS)
def test_backward_after_the_module_is_gone(mods, oracle, kind):
    p = Pair(mods, oracle, kind)
    rng = np.random.default_rng(9)
    batch = p.draw(rng, 48)
    coefs = _coef(rng, 48, p.tables)
    loss = _loss(p.forward(batch), coefs)
    p.mod = p.param = p.o_gpu = None
    gc.collect()
    loss.backward()
    p.push(batch, coefs)
    p.check("after a backward without its module")


@pytest.mark.parametrize("kind", KINDS)
def test_contiguous_gradient_off_its_alignment(mods, oracle, kind):
    """A batch of one behind 13 dense features: what torch.cat hands back for an embedding is one row
    that starts 13 floats into the matrix, contiguous and not on a 16-byte boundary."""
    p = Pair(mods, oracle, kind)
    rng = np.random.default_rng(3)
    for _ in range(2):
        batch = p.draw(rng, 1)
        outs = p.forward(batch)
        seen = []
        for o in outs:
            o.register_hook(lambda g: seen.append((g.is_contiguous(), g.data_ptr() % 16)))
        dense = torch.ones((1, 13), device="cuda")
        coef = (rng.integers(-8, 9, size=(1, 13 + DIM * len(outs))) / 16.0).astype(np.float32)
        (torch.cat([dense] + list(outs), dim=1) * torch.from_numpy(coef).cuda()).sum().backward()
        assert seen and all(c and off for c, off in seen)       # the form this test is about
        p.push(batch, [coef[:, 13 + DIM * i:13 + DIM * (i + 1)] for i in range(len(outs))])
    p.check("after gradients at odd addresses")


class _NoGradient(torch.autograd.Function):
    """A function whose backward has no gradient to hand on."""

    @staticmethod
    def forward(ctx, x):
        return x.clone()

    @staticmethod
    def backward(ctx, grad):
        return None


@pytest.mark.parametrize("kind", KINDS)
def test_undefined_gradient_pushes_zeros(mods, oracle, kind):
    p = Pair(mods, oracle, kind)
    rng = np.random.default_rng(2)
    for step in range(3):
        batch = p.draw(rng, 64)
        outs = p.forward(batch)
        coefs = _coef(rng, 64, p.tables)
        if step == 1:
            sum(_NoGradient.apply(o).sum() for o in outs).backward()
            coefs = [np.zeros_like(c) for c in coefs]
        else:
            _loss(outs, coefs).backward()
        p.push(batch, coefs)
    p.check("after a step without gradients")


@pytest.mark.parametrize("kind", KINDS)
def test_ids_unpacked_by_hooks_are_looked_up_again(mods, oracle, kind):
    """Saved-tensor hooks that offload to the host and bring every tensor back into one buffer per
    shape: the first backward gets its ids at the address, and in the number, that the second forward
    pulled from."""
    p = Pair(mods, oracle, kind, (3, {}))
    rng = np.random.default_rng(6)
    first = p.draw(rng, 64, span=100)
    # the same bags, other ids
    second = [((ids + np.uint64(100)), off) for ids, off in first]
    own, shared = p.tensors(first), p.tensors(second)
    buffers = [t for pair in shared for t in pair if t is not None]
    packed = []

    def pack(t):
        packed.append(t)
        i = (len(packed) - 1) % len(order)
        return order[i], t.cpu()

    def unpack(x):
        b = buffers[x[0]]
        b.copy_(x[1])
        return b

    # modules save ids (and offsets) of all tables in one order: all ids, then all offsets
    order = list(range(len(buffers))) if p.tables == 1 or not p.jagged else [0, 2, 1, 3]
    with torch.autograd.graph.saved_tensors_hooks(pack, unpack):
        outs_a = p.forward(first, own)
        outs_b = p.forward(second, shared)
    assert len(packed) == 2 * len(order)
    ca, cb = _coef(rng, 64, p.tables), _coef(rng, 64, p.tables)
    _loss(outs_a, ca).backward()
    _loss(outs_b, cb).backward()
    p.push(first, ca)
    p.push(second, cb)
    p.check("after two backward passes through one buffer")


@pytest.mark.parametrize("kind", KINDS)
def test_expanded_gradient(mods, oracle, kind):
    """The gradient of a plain sum is one value expanded over the output; that of a sum over the batch is
    one row, read by every position."""
    p = Pair(mods, oracle, kind)
    rng = np.random.default_rng(10)
    row = (np.arange(DIM, dtype=np.float32) - 8) / 16
    for step in range(4):
        batch = p.draw(rng, 40)
        outs = p.forward(batch)
        seen = []
        for o in outs:
            o.register_hook(lambda g: seen.append(g.stride()[0]))
        if step % 2:
            sum(o.sum() for o in outs).backward()
            want = np.ones((40, DIM), np.float32)
        else:
            sum((o.sum(dim=0) * torch.from_numpy(row).cuda()).sum() for o in outs).backward()
            want = np.tile(row, (40, 1))
        assert seen == [0] * len(outs)
        p.push(batch, [want] * len(outs))
    p.check("after expanded gradients")


@pytest.mark.parametrize("kind", KINDS)
def test_backward_twice_over_a_retained_graph(mods, oracle, kind):
    """Every backward pushes; without retain_graph a second one is refused."""
    p = Pair(mods, oracle, kind)
    rng = np.random.default_rng(11)
    batch = p.draw(rng, 48)
    coefs = _coef(rng, 48, p.tables)
    loss = _loss(p.forward(batch), coefs)
    loss.backward(retain_graph=True)
    p.push(batch, coefs)
    loss.backward()
    p.push(batch, coefs)
    with pytest.raises(RuntimeError, match="second time"):
        loss.backward()
    p.check("after two backward passes")


@pytest.mark.parametrize("kind", KINDS)
def test_saved_tensors_on_the_host(mods, oracle, kind):
    p = Pair(mods, oracle, kind)
    rng = np.random.default_rng(12)
    for _ in range(2):
        batch = p.draw(rng, 48)
        coefs = _coef(rng, 48, p.tables)
        with torch.autograd.graph.save_on_cpu():
            loss = _loss(p.forward(batch), coefs)
        loss.backward()
        p.push(batch, coefs)
    p.check("after backward passes over saved tensors from the host")


def test_pooled_request_a_table_at_a_time(mods, oracle):
    """A request above what one combined call takes goes through the tables' own calls, forward and
    backward, with an output that has no gradient among them, and may change from step to step."""
    p = Pair(mods, oracle, "combine_jagged", (1, {}))
    rng = np.random.default_rng(13)
    limit = p.param._native.combined_max
    for step in range(4):
        p.param._native.combined_max = 50 if step in (1, 2) else limit
        batch = p.draw(rng, 64)
        outs = p.forward(batch)
        coefs = _coef(rng, 64, 2)
        _loss(outs, [coefs[0], None if step == 2 else coefs[1]]).backward()
        p.push(batch, [coefs[0], np.zeros_like(coefs[1]) if step == 2 else coefs[1]])
    p.check("after requests of both kinds")


def test_pooled_push_whose_keys_do_not_fit_goes_a_table_at_a_time(mods, oracle):
    """32 tables of which one has room for more than 2^26 rows: member and row number take 33 bits, and
    the combined push answers that it cannot (KRK_E_CAPACITY)."""
    api, te = mods
    n_tables, dim = 32, 4
    init = api.Initializer.create(api.InitializerType.kConstant, {"value": "1"})
    emb = te.CombineJaggedEmbedding([dim] * n_tables, [init] * n_tables, optim=api.Optim.create(api.OptimType.kSGD),
                                    lr=0.5)
    emb.combine_sparse_table.tables()[3].reserve((1 << 26) + 1)
    rng = np.random.default_rng(14)
    ids = [rng.integers(0, 50, size=60) for _ in range(n_tables)]
    off = torch.arange(0, 61, 3).cuda()                  # 20 bags of three
    outs = emb([te.JaggedTensor(torch.from_numpy(i).cuda(), off) for i in ids])
    assert all(torch.equal(o, torch.full((20, dim), 3.0, device="cuda")) for o in outs)
    group = emb.combine_sparse_table._groups[dim]
    assert group.CombinePushRaw(emb.combine_sparse_table._optim, np.concatenate(ids).astype(np.uint64),
                                np.arange(0, 60 * n_tables + 1, 60), np.zeros((60 * n_tables, dim), np.float32),
                                0.5) == api.E_CAPACITY
    sum(o.sum() for o in outs).backward()
    torch.cuda.synchronize()
    for i, t in zip(ids, emb.combine_sparse_table.tables()):
        u, count = np.unique(i, return_counts=True)
        want = 1.0 - 0.5 * count.astype(np.float32)
        assert np.array_equal(t.Pull(u.astype(np.uint64))[1], np.repeat(want[:, None], dim, axis=1))
