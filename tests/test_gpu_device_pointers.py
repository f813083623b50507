"""Caller memory of every kind at the entry points that take device pointers."""
import ctypes

import numpy as np
import pytest

from helpers import random_cell

pytestmark = pytest.mark.gpu

RC = 4.0


class Memory:
    """Arrays in device or pinned host memory, by the HIP runtime itself."""

    def __init__(self):
        self.hip = ctypes.CDLL("libamdhip64.so")
        p, n = ctypes.c_void_p, ctypes.c_size_t
        for fn, args in (("hipMalloc", [ctypes.POINTER(p), n]), ("hipFree", [p]),
                         ("hipHostMalloc", [ctypes.POINTER(p), n, ctypes.c_uint]),
                         ("hipHostFree", [p]), ("hipMemcpy", [p, p, n, ctypes.c_int])):
            getattr(self.hip, fn).argtypes = args
        self.held = []

    def get(self, size, pinned=False):
        p = ctypes.c_void_p()
        if pinned:
            assert self.hip.hipHostMalloc(ctypes.byref(p), size, 0) == 0
        else:
            assert self.hip.hipMalloc(ctypes.byref(p), size) == 0
        self.held.append((p, pinned))
        return p.value

    def put(self, p, a, size=None):
        assert self.hip.hipMemcpy(p, a.ctypes.data, size or a.nbytes, 4) == 0

    def read(self, p, a):
        assert self.hip.hipMemcpy(a.ctypes.data, p, a.nbytes, 4) == 0
        return a

    def free(self):
        for p, pinned in self.held:
            assert (self.hip.hipHostFree if pinned else self.hip.hipFree)(p) == 0


@pytest.fixture
def memory():
    m = Memory()
    yield m
    m.free()


@pytest.fixture(scope="module")
def system():
    return random_cell(50, 5, nos=2, scale=8.8, skew=0.2)


def neighbors(h):
    from flare_amd import _lib
    L = _lib.load()
    sweep, nnb, vol, ssc = ctypes.c_int(), ctypes.c_int64(), ctypes.c_double(), ctypes.c_double()
    _lib.check(L.fm_structure_info(h, ctypes.byref(sweep), ctypes.byref(nnb), ctypes.byref(vol),
                                   ctypes.byref(ssc)))
    sp, rel = np.zeros(nnb.value, np.int32), np.zeros((nnb.value, 4))
    _lib.check(L.fm_structure_get_neighbors(h, None, None, None, None, _lib.ptr(sp),
                                            _lib.ptr(rel)))
    _lib.check(L.fm_structure_destroy(h))
    return sp, rel


def create(fn, system, species, positions):
    from flare_amd import _lib
    h = ctypes.c_void_p()
    cell = _lib.f64(system[0].reshape(-1))
    rc = getattr(_lib.load(), fn)(_lib.default_context().h, _lib.ptr(cell), len(system[1]),
                                  species, positions, RC, ctypes.byref(h))
    return rc, h


@pytest.mark.parametrize("kind", ["device", "slice", "misaligned", "pinned"])
def test_structure_sources(system, memory, kind):
    """Species and positions in the GPU's memory, inside a larger array, at an
    address that is no multiple of the element's size, and in pinned memory."""
    from flare_amd import _lib
    arrays = [_lib.i32(system[1]), _lib.f64(system[2]).reshape(-1)]
    rc, h = create("fm_structure_create", system, *map(_lib.ptr, arrays))
    _lib.check(rc)
    want = neighbors(h)
    lead = {"device": 0, "slice": 16, "misaligned": 2, "pinned": 0}[kind]
    ptrs = [memory.get(lead + a.nbytes, kind == "pinned") + lead for a in arrays]
    for p, a in zip(ptrs, arrays):
        memory.put(p, a)
    rc, h = create("fm_structure_create_device", system, *ptrs)
    _lib.check(rc)
    got = neighbors(h)
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])


@pytest.mark.parametrize("short", [0, 1])
def test_short_array(system, memory, short):
    """An array shorter than the atom count is an error, as for a copy, and the
    next structure is built as if it had not been."""
    from flare_amd import _lib
    arrays = [_lib.i32(system[1]), _lib.f64(system[2]).reshape(-1)]
    rc, h = create("fm_structure_create", system, *map(_lib.ptr, arrays))
    _lib.check(rc)
    want = neighbors(h)
    sizes = [a.nbytes - (16 if k == short else 0) for k, a in enumerate(arrays)]
    ptrs = [memory.get(size) for size in sizes]
    for p, a, size in zip(ptrs, arrays, sizes):
        memory.put(p, a, size)
    for _ in range(5):
        rc, h = create("fm_structure_create_device", system, *ptrs)
        assert rc == _lib.FM_ERR_HIP
        rc, h = create("fm_structure_create", system, *map(_lib.ptr, arrays))
        _lib.check(rc)
        got = neighbors(h)
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])


@pytest.mark.parametrize("reps", [2, 15])
@pytest.mark.parametrize("where", ["device", "pinned", "mixed"])
def test_prediction_outputs(memory, reps, where):
    """Results in device and in pinned memory, small ones (which reach pageable
    memory through a staging buffer) and large ones."""
    from flare_amd import _C_flare as C
    from flare_amd import _lib
    from helpers import fcc
    calc = C.B2("chebyshev", "quadratic", [0.0, RC], [], [1, 4, 2])
    train = C.Structure(*fcc(4.0, (3, 3, 3), 0.1, 3), RC, [calc])
    sgp = C.SparseGP([C.NormalizedDotProduct(1.5, 2.0)], 0.1, 0.1, 0.1)
    sgp.add_specific_environments(train, [0, 9, 40])
    sgp.update_L_inverse()
    sgp.set_alpha(np.linspace(0.2, 0.5, sgp.n_sparse))
    s = C.Structure(*fcc(4.0, (reps,) * 3, 0.1, 4), RC, [calc])
    sizes = (1 + 3 * s.noa + 6, s.noa, s.noa)
    model = sgp._model(0, s._ctx)

    def predict(ptrs):
        _lib.check(_lib.load().fm_predict(model.h, s._h, _lib.PREDICT_MEAN | _lib.PREDICT_LOCAL,
                                          0, *ptrs))

    want = [np.zeros(k) for k in sizes]
    predict([_lib.ptr(w) for w in want])
    assert (sum(sizes) * 8 > 256 << 10) == (reps == 15)
    out = [np.zeros(k) for k in sizes]
    ptrs = [_lib.ptr(o).value if where == "mixed" and k != 1
            else memory.get(8 * sizes[k], where == "pinned") for k, o in enumerate(out)]
    predict(ptrs)
    for k, (p, o) in enumerate(zip(ptrs, out)):
        if p != o.ctypes.data:
            memory.read(p, o)
        assert np.array_equal(o, want[k])
