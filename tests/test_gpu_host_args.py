"""Arguments in pageable host memory. Up to 1 MB they pass through page-locked buffers, which the kernels
read in place or, where they read them several times over or out of order, from a copy on the device.
Which of the two it is depends on sizes; sizes on either side of the rule (and sizes that are no whole
number of 16-byte vectors) give what device arrays give, to the bit: gradients and weights are dyadic, so that
sums do not depend on their order, which the numbers of the rows decide."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

READ_AGAIN = 128 << 10      # bytes read beyond the argument's own from which it is copied
PIECE = 128                 # a read across PCIe counts at least as much


@pytest.fixture(scope="module")
def api():
    from kraken_amd import api as a
    a.lib()
    return a


def _pair(api, dim):
    init = api.Initializer.create(api.InitializerType.kNormal, {"stddev": "0.01", "seed": "5"})
    return api.SparseTable(dim, init), api.SparseTable(dim, init)


def _same(a, b):
    ia, va, _, _ = a.export()
    ib, vb, _, _ = b.export()
    oa, ob = np.argsort(ia), np.argsort(ib)
    assert np.array_equal(ia[oa], ib[ob]) and np.array_equal(va[oa], vb[ob])


def _edge(bytes_, piece):
    """the smallest number of reads of `piece` bytes for which an argument of `bytes_` is copied"""
    return -(-(bytes_ + READ_AGAIN) // max(piece, PIECE))


def _dyadic(rng, shape):
    return (rng.integers(-8, 9, size=shape) / 16.0).astype(np.float32)


@pytest.mark.parametrize("mode,weighted", [("sum", False), ("mean", False), ("mean", True)])
@pytest.mark.parametrize("dim,bags", [(16, 512), (5, 701), (64, 300), (128, 77)])
def test_pooled_push_from_pageable_memory(api, dim, bags, mode, weighted):
    rng = np.random.default_rng(dim + bags)
    host, dev = _pair(api, dim)
    opt = api.Optim.create(api.OptimType.kSGD)
    edge = max(_edge(bags * dim * 4, dim * 4), bags + 1)
    # a mean of a power of two of ids is dyadic: bags of equal length then, and the sizes of the sum
    # on both sides of the rule; the largest take the sorted path
    sizes = (edge - 1, edge, edge + 1234, 20_001) if mode == "sum" else [bags * 2 ** k for k in (0, 1, 2, 3, 6)]
    for n in sizes:
        ids = rng.integers(0, 900, size=n).astype(np.uint64)
        cuts = np.sort(rng.integers(0, n + 1, size=bags - 1)) if mode == "sum" else np.arange(1, bags) * (n // bags)
        off = np.concatenate([[0], cuts, [n]]).astype(np.int64)
        g = _dyadic(rng, (bags, dim))
        w = (2.0 ** rng.integers(-1, 2, size=n)).astype(np.float32) if weighted else None
        d = api.DeviceArray.from_host
        seen = np.unique(ids)
        assert host.Pull(seen)[0] == 0 and dev.Pull(d(seen))[0] == 0
        assert host.PushPooled(opt, ids, off, g, 0.5, mode=mode, weights=w) == 0
        assert dev.PushPooled(opt, d(ids), d(off), d(g), 0.5, mode=mode, weights=None if w is None else d(w)) == 0
        _same(host, dev)


@pytest.mark.parametrize("dim", [8, 5, 32])
def test_push_raw_from_pageable_memory(api, dim):
    rng = np.random.default_rng(dim)
    host, dev = _pair(api, dim)
    g_host, g_dev = api.TableGroup([host]), api.TableGroup([dev])
    opt = api.Optim.create(api.OptimType.kSGD)
    edge = READ_AGAIN // (PIECE - 4 * dim) if 4 * dim < PIECE else 1500
    for n in (edge - 3, edge + 3, 14_001 if 14_001 * dim * 4 <= 1 << 20 else 8190):
        ids = rng.integers(0, 700, size=n).astype(np.uint64)
        g = _dyadic(rng, (n, dim))
        d_ids, d_g = api.DeviceArray.from_host(ids), api.DeviceArray.from_host(g)
        off = np.array([0, n], np.int64)
        seen = np.unique(ids)
        assert host.Pull(seen)[0] == 0 and dev.Pull(api.DeviceArray.from_host(seen))[0] == 0
        assert host.PushRaw(opt, ids, g, 0.5) == 0 and dev.PushRaw(opt, d_ids, d_g, 0.5) == 0
        _same(host, dev)
        assert g_host.CombinePushRaw(opt, ids, off, g, 0.5) == 0
        assert g_dev.CombinePushRaw(opt, d_ids, off, d_g, 0.5) == 0
        _same(host, dev)


@pytest.mark.parametrize("n", [1021, READ_AGAIN // 16 - 1, READ_AGAIN // 16 + 1, READ_AGAIN // 4 + 3, 262_143])
def test_codec_step_from_pageable_memory(api, n):
    """a selecting call reads the gradient five times, another one twice"""
    rng = np.random.default_rng(n)
    host, dev = api.DenseBag(n), api.DenseBag(n)
    for _ in range(3):                                   # the first step of three selects
        g = rng.standard_normal(n).astype(np.float32)
        idx, val = host.MaybeToCoo(3, 0.75, g)
        d_idx, d_val, nnz = dev.MaybeToCoo(3, 0.75, api.DeviceArray.from_host(g))
        assert nnz == idx.size
        assert np.array_equal(d_idx.to_host()[:nnz], idx) and np.array_equal(d_val.to_host()[:nnz], val)
        assert np.array_equal(host.residual, dev.residual) and host.tau == dev.tau
