"""The native launch route (csrc/py/launch.cpp) against the ctypes one: the same descriptors for every form of tensor it
takes, nothing called for the forms it leaves, and the same errors."""
import ctypes
import threading
import time

import pytest
import torch


class _Sub(torch.Tensor):
    pass


def _left_alone():
    t = torch.zeros(4)
    return [torch.zeros(1, 1, 1, 1, 1), torch.zeros(3, dtype=torch.bool), torch.zeros(3, dtype=torch.complex64),
            torch.zeros(3).as_subclass(_Sub), torch.eye(3).to_sparse(), t.numpy(), [1.0], 3]


@pytest.mark.parametrize("i", range(8))
def test_other_arguments_are_left_to_ctypes(ct, i):
    ct.lib()
    assert ct._native.mi_vec_add_kernel_1d(_left_alone()[i], None, None, 16, None) is None


@pytest.mark.parametrize("tile", [1.0, "16", 2 ** 31, -2 ** 31 - 1, None])
def test_other_numbers_are_left_to_ctypes(ct, tile):
    ct.lib()
    assert ct._native.mi_vec_add_kernel_1d(None, None, None, tile, None) is None


def test_wrong_number_of_arguments_is_left_to_ctypes(ct):
    ct.lib()
    assert ct._native.mi_vec_add_kernel_1d(None, None, 16, None) is None


@pytest.fixture
def unloaded(ct, monkeypatch):
    """The package as before its first call, with a stream look-up that needs no GPU."""
    ct.lib()
    for name, value in (("_lib", None), ("_native", None), ("_streams", False), ("_stream", lambda stream=None: ctypes.c_void_p(0))):
        monkeypatch.setattr(ct, name, value)
    return ct


def _empty_call(ct):
    e = torch.zeros(0)
    ct.vec_add_kernel_1d(e, e, e, 16)   # (nothing to do: MI_OK before any GPU call)


def test_first_calls_from_several_threads(unloaded, monkeypatch):
    """Calls that come while the first one is still loading the library."""
    ct, load, errors = unloaded, unloaded._load_native, []
    monkeypatch.setattr(ct, "_load_native", lambda cdll: (time.sleep(0.2), load(cdll))[1])

    def work():
        try:
            for _ in range(20):
                _empty_call(ct)
        except Exception as e:   # noqa: BLE001
            errors.append(e)
    threads = [threading.Thread(target=work) for _ in range(8)]
    for t in threads:
        t.start()
        time.sleep(0.01)
    for t in threads:
        t.join()
    assert not errors and ct._native is not None


def test_a_missing_library_is_named_by_every_call(unloaded, monkeypatch):
    monkeypatch.setattr(unloaded, "LIB_PATH", "/nowhere/libmi355tile.so")
    for _ in range(3):
        with pytest.raises(RuntimeError, match="/nowhere/libmi355tile.so is missing"):
            _empty_call(unloaded)


def test_without_the_module_launches_take_the_ctypes_route(unloaded, monkeypatch):
    monkeypatch.setattr(unloaded, "_native_path", lambda: "/nowhere/launch.so")
    with pytest.warns(RuntimeWarning, match="/nowhere/launch.so is missing"):
        _empty_call(unloaded)
    _empty_call(unloaded)
    assert unloaded._native is None
    with pytest.raises(unloaded.MiError):
        unloaded.vec_add_kernel_1d(torch.zeros(0), torch.zeros(0), torch.zeros(0), 7)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["float32", "float64", "float16", "bfloat16", "int32", "int64", "float8_e4m3fn", "float8_e5m2"])
def test_descriptors_are_those_of_the_ctypes_route(ct, dtype):
    dt = getattr(torch, dtype)
    base = torch.zeros(3, 5, 4, 8, dtype=torch.float32, device="cuda").to(dt)
    forms = [base, base[0], base[:, 1:3, ::2, 3:7], base.transpose(0, 3), base[0, 0].t(), base[0, 0, 0, 0], base[:0],
             base[0, 0, 0].expand(6, 8), torch.nn.Parameter(base, requires_grad=False)]
    seen = []
    proto = ctypes.CFUNCTYPE(ctypes.c_int, *ct._SIGNATURES["mi_layer_norm_fwd"][0])

    def record(*args):
        seen.append(([None if not a else bytes(a.contents) for a in args[:6]], args[6], args[7], args[8]))
        return 7
    cb = proto(record)
    table = {n: ctypes.cast(getattr(ct.lib(), n), ctypes.c_void_p).value for n in ct._SIGNATURES}
    ct._native.bind_library({**table, "mi_layer_norm_fwd": ctypes.cast(cb, ctypes.c_void_p).value})
    side = torch.cuda.Stream()
    try:
        for f in forms:
            with torch.cuda.stream(side):
                assert ct._native.mi_layer_norm_fwd(f, None, f, f, f, f, 1e-5, -3, None) == 7
    finally:
        ct._native.bind_library(table)
    assert len(seen) == len(forms)
    for f, (arrays, eps, tile, stream) in zip(forms, seen):
        want = bytes(ct.TileArray(f))
        assert arrays == [want, None, want, want, want, want]
        assert eps == ctypes.c_float(1e-5).value and tile == -3 and stream == side.cuda_stream


@pytest.mark.gpu
def test_errors_are_those_of_the_ctypes_route(ct):
    a = torch.zeros(8, device="cuda")
    ct.vec_add_kernel_1d(a, a, a, 8)
    with pytest.raises(TypeError):
        ct.vec_add_kernel_1d(a, a, a.bool(), 8)
    with pytest.raises(ValueError):
        ct.vec_add_kernel_1d(a, a, a.view(1, 1, 1, 1, 8), 8)
    with pytest.raises(ctypes.ArgumentError):
        ct.vec_add_kernel_1d(a, a, a, 8.0)
    with pytest.raises(ct.MiError) as e:
        ct.vec_add_kernel_1d(a, a, a[:4], 7)
    with pytest.raises(ct.MiError) as e2:
        ct.vec_add_kernel_1d(a, a, a[:4], 7, stream=torch.cuda.current_stream())
    assert e.value.code == e2.value.code
