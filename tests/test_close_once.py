"""Closing a context or a server from several threads (a thread's own close, a
last reference dropped elsewhere, the exit hook): the library's destroy is
called once, and no close returns before it has ended.  On the CPU, with a
library that only counts."""
import ctypes
import threading
import types

import pytest

import kamsta_amd as k


@pytest.mark.parametrize("cls,entry", [(k.Context, "kmst_context_destroy"),
                                       (k.Server, "kmst_server_destroy")])
def test_one_destroy_for_closes_from_two_threads(monkeypatch, cls, entry):
    inside, leave, destroyed, ended = threading.Event(), threading.Event(), [], []

    def destroy(h):
        destroyed.append(ctypes.cast(h, ctypes.c_void_p).value)
        inside.set()
        assert leave.wait(30)
        ended.append(1)

    def create(*args):
        args[-1]._obj.value = 4096
        return k.KMST_OK

    lib = types.SimpleNamespace(**{entry: destroy, "kmst_context_create": create,
                                   "kmst_server_create": create,
                                   "kmst_server_config_default": lambda c: None})
    monkeypatch.setattr(k, "load", lambda: lib)
    obj = cls()
    after = []  # destroys that had ended when the second close returned
    first = threading.Thread(target=obj.close)
    second = threading.Thread(target=lambda: (obj.close(), after.append(len(ended))))
    first.start()
    assert inside.wait(30)
    second.start()
    second.join(0.2)
    leave.set()
    first.join(30)
    second.join(30)
    obj.close()
    assert destroyed == [4096]
    assert after == [1]
