"""CPU-side checks of the C ABI: the library loads, exports every symbol the header declares,
parses optimizer/initializer confs like the reference, and refuses to run without a GPU."""
import ctypes as C
import os
import re

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def api():
    from kraken_amd import api as a
    if not os.path.exists(a.LIB_PATH):
        from kraken_amd import build
        build.build(verbose=False)
    a.lib()
    return a


def test_every_declared_symbol_is_exported(api):
    header = open(os.path.join(ROOT, "include", "kraken_hip.h")).read()
    names = sorted(set(re.findall(r"\b(krk_[a-z0-9_]+)\s*\(", header)))
    assert len(names) > 40
    L = C.CDLL(api.LIB_PATH)
    missing = [n for n in names if not hasattr(L, n)]
    assert not missing, missing
    # and the binding knows every one of them
    assert not [n for n in names if n not in api.EXPORTS]


def test_flag_bits_of_the_binding_are_the_headers(api):
    """The call flags are single, distinct bits, and the ctypes binding carries the header's values."""
    header = open(os.path.join(ROOT, "include", "kraken_hip.h")).read()
    flags = {n: int(v, 16) for n, v in re.findall(r"#define (KRK_(?:DEVICE_PTRS|ASYNC|NOTE_ROWS|IDS_AS_PULLED)) (0x[0-9a-f]+)u", header)}
    assert flags == {"KRK_DEVICE_PTRS": api.DEVICE_PTRS, "KRK_ASYNC": api.ASYNC, "KRK_NOTE_ROWS": api.NOTE_ROWS,
                     "KRK_IDS_AS_PULLED": api.IDS_AS_PULLED}
    bits = sorted(flags.values())
    assert all(b and b & (b - 1) == 0 for b in bits) and len(set(bits)) == len(bits)


def test_optim_conf_parsing_matches_oracle_defaults(api, oracle):
    """Optim::Create (ps/optim/optim.cc:18-105): defaults and has_* flags."""
    for type_ in (0, 1, 2, 3):
        g = api.Optim.create(type_).raw
        r = oracle.optim(type_)
        for f in ("type", "has_weight_decay", "weight_decay", "has_momentum", "momentum",
                  "has_dampening", "dampening", "nesterov", "beta1", "beta2", "eps", "amsgrad",
                  "alpha", "centered"):
            assert getattr(g, f) == getattr(r, f), (type_, f)
        assert g.initial_accumulator == 0.0
    g = api.Optim.create(3, {"weight_decay": "0.5", "momentum": "0.9", "dampening": "0.1",
                             "nesterov": "TRUE", "eps": "3"}).raw
    assert (g.has_weight_decay, g.has_momentum, g.has_dampening, g.nesterov) == (1, 1, 1, 1)
    assert g.eps == np.float32(1e-8)                 # SGD has no eps key
    g = api.Optim.create(1, {"amsgrad": "1", "beta1": "oops", "beta2": "0.5"}).raw
    assert g.amsgrad == 1 and g.beta1 == np.float32(0.9) and g.beta2 == np.float32(0.5)
    g = api.Optim.create(2, {"centered": "yes", "alpha": "0.9"}).raw
    assert g.centered == 0 and g.alpha == np.float32(0.9)   # only "true"/"1" are true (utils.h:83-87)
    assert api.Optim.create(4) is None


def test_initializer_conf_parsing(api):
    """Initializer::Create (ps/initializer/initializer.cc:22-61) defaults and keys."""
    I = api.Initializer
    assert (I.create(0).raw.a, I.create(0, {"value": "2.5"}).raw.a) == (0.0, 2.5)
    u = I.create(1).raw
    assert (u.a, u.b) == (0.0, 1.0)
    n = I.create(2, {"mean": "1", "stddev": "0.01", "seed": "7"}).raw
    assert (n.a, n.b, n.seed) == (1.0, np.float32(0.01), 7)
    assert I.create(3).raw.a == 1.0 and I.create(4, {"gain": "2"}).raw.a == 2.0
    assert I.create(5) is None


def test_error_messages(api):
    L = api.lib()
    assert L.krk_error_message(0) == b"Success"
    assert L.krk_error_message(12) == b"SparseId not exist"
    assert L.krk_error_message(11) == b"Uncompatible gradient"


def test_no_gpu_fails_loudly(api):
    """Without a GPU every object constructor fails with a device error; nothing computes on CPU."""
    L = api.lib()
    cnt = C.c_int()
    try:
        hip = C.CDLL("libamdhip64.so")
        have_gpu = hip.hipGetDeviceCount(C.byref(cnt)) == 0 and cnt.value > 0
    except OSError:
        have_gpu = False
    if have_gpu:
        pytest.skip("a GPU is present")
    with pytest.raises(api.KrakenHipError) as e:
        api.SparseTable(8, api.Initializer.create(0))
    assert e.value.code == api.E_DEVICE
    with pytest.raises(api.KrakenHipError):
        api.DenseTable(np.zeros(4, np.float32))
    with pytest.raises(api.KrakenHipError):
        api.DenseBag(1024)
    with pytest.raises(api.KrakenHipError):
        api.dedup(np.arange(4, dtype=np.uint64))


@pytest.mark.parametrize("form", ["plain", "view", "read_only", "strided", "fortran", "empty", "records", "dates", "scalar"])
def test_an_array_argument_is_its_address(api, form):
    """Whichever way api._ptr gets at an array's address: it is numpy's, and the argument keeps the array."""
    import gc
    import weakref
    make = {"plain": lambda: np.arange(12, dtype=np.uint64), "view": lambda: np.zeros((5, 6), np.float32)[2:],
            "read_only": lambda: np.frombuffer(b"abcdefgh", np.uint8), "strided": lambda: np.zeros((4, 6), np.float32)[:, 1::2],
            "fortran": lambda: np.zeros((4, 6), np.float32, order="F"), "empty": lambda: np.zeros((0, 4), np.float32),
            "records": lambda: np.zeros(3, [("rank", "<u8"), ("dim", "u1")]), "dates": lambda: np.zeros(3, "datetime64[s]"),
            "scalar": lambda: np.zeros((), np.float32)}[form]
    a = make()
    arg = api._ptr(a)
    assert form == "empty" or C.cast(arg, C.c_void_p).value == a.ctypes.data
    alive = weakref.ref(a)
    del a
    gc.collect()
    assert alive() is not None
    del arg
    gc.collect()
    assert alive() is None
    assert api._ptr(None) is None


@pytest.mark.parametrize("make", [lambda: bytearray(64), lambda: memoryview(bytearray(64)), lambda: (C.c_float * 16)(),
                                  lambda: __import__("array").array("f", [0.0] * 16), lambda: [0.0] * 16, lambda: b"0" * 64])
def test_what_is_no_array_is_refused(api, make):
    """Buffers of other kinds carry neither shape nor type: an `out` of the wrong length would be written past its end."""
    with pytest.raises(AttributeError):
        api._ptr(make())


def test_arrays_of_two_kinds_in_one_call(api):
    """Device arrays in a call say so in its flags, and are not mixed with host arrays."""
    dev = api.DeviceArray.__new__(api.DeviceArray)
    dev.ptr = None
    host = np.zeros(3, np.float32)
    assert api._flags() == 0 and api._flags(None, extra=api.ASYNC) == api.ASYNC
    assert api._flags(host, None) == 0
    assert api._flags(dev, None, dev, extra=api.ASYNC) == api.DEVICE_PTRS | api.ASYNC
    for arrays in ((dev, host), (host, dev), (None, host, dev)):
        with pytest.raises(ValueError):
            api._flags(*arrays)


def test_lanes_meet_in_lds_in_order():
    """Where lanes of a wavefront pass words to each other through LDS without a workgroup's barrier, fences stand around
    the wavefront's barrier, which is no access to memory to the compiler: krk_internal.h's wave_lds_order."""
    import glob
    csrc = os.path.join(ROOT, "kraken_amd", "csrc")
    uses = [(os.path.basename(p), line.strip()) for p in sorted(glob.glob(os.path.join(csrc, "*")))
            for line in open(p) if "amdgcn_wave_barrier" in line]
    assert uses == [("krk_internal.h", "__builtin_amdgcn_wave_barrier();")]
    inline = open(os.path.join(csrc, "krk_internal.h")).read().split("void wave_lds_order() {")[1].split("}")[0].split()
    assert inline == ['__builtin_amdgcn_fence(__ATOMIC_RELEASE,', '"wavefront");', "__builtin_amdgcn_wave_barrier();",
                      '__builtin_amdgcn_fence(__ATOMIC_ACQUIRE,', '"wavefront");']
