"""The tests that name a kernel (conftest.NAMED_KERNELS) on the kernels that a caller gets: every comparison of values that they hold,
at their sizes.  Each body runs twice, first with its kernel chosen as in its own file, noting the names that it is given, then with
nothing switched off and the same names handed to it, so that only its checks of names are met from the first run."""
import importlib
import inspect
import threading

import pytest

pytest.importorskip("torch")

from conftest import NAMED_KERNELS, switches_of

pytestmark = pytest.mark.gpu

HOME = {name: file for files in NAMED_KERNELS.values() for file, names in files.items() for name in names}
globals().update({name: getattr(importlib.import_module(file), name) for name, file in HOME.items()})


# test -> for each of its parameters, whether it ran other kernels than those that it names
seen = {}


@pytest.fixture(autouse=True)
def _values_of_the_default_route(request, ct):
    name = request.function.__name__
    if name not in HOME:
        yield
        return
    real, noted, given, other = ct.last_variant, [], [], {}

    def note():
        noted.append(real())
        return noted[-1]

    def hand_out():
        now = real()
        if threading.current_thread() is not threading.main_thread():   # (threads repeat what the main one has done)
            return other.get(now, now)
        given.append(now)
        other[now] = noted[len(given) - 1]
        return other[now]

    params = getattr(request.node, "callspec", None)
    with pytest.MonkeyPatch.context() as first:
        for switch in switches_of(HOME[name], name):
            first.setenv(switch, "0")
        first.setattr(ct, "last_variant", note)
        args = {n: first if n == "monkeypatch" else params.params[n] if params and n in params.params else request.getfixturevalue(n)
                for n in inspect.signature(request.function).parameters}
        request.function(**args)
    with pytest.MonkeyPatch.context() as second:
        second.setattr(ct, "last_variant", hand_out)
        yield
    seen.setdefault(name, []).append(given != noted)


def test_zz_each_of_them_was_on_another_kernel():
    """(last in the file; only what was run counts)"""
    assert all(any(v) for v in seen.values()), [n for n, v in seen.items() if not any(v)]
