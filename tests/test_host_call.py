"""The native side of a launch (`csrc/host_call.cpp`) without a GPU: arguments, refusals, recording and making again.  The functions
called are Python's own, by way of ctypes callbacks."""
import ctypes
from ctypes import c_double, c_float, c_int, c_int64, c_void_p

import numpy as np
import pytest
import torch

from minfer_amd.kernels import build, ops

_TYPES = {"p": c_void_p, "i": c_int, "q": c_int64, "f": c_float, "d": c_double}


class Calls:
    """A `Launch` on a function of these argument kinds that notes what it was called with and returns `rc`."""

    def __init__(self, kinds, recorded=False):
        self.seen, self.rc = [], 0

        def note(*args):
            self.seen.append(args)
            return self.rc
        self._keep = ctypes.CFUNCTYPE(c_int, *[_TYPES[k] for k in kinds])(note)
        self.launch = build.load_extension("host_call").Launch(ctypes.cast(self._keep, c_void_p).value, kinds, recorded)


def record():
    return build.load_extension("host_call").Record()


def test_arguments_arrive_as_they_are():
    c = Calls("pipqfdpi")
    t = torch.zeros(4)
    ints = (c_int * 3)(1, 2, 3)
    assert c.launch(t, -5, None, -(1 << 40), 0.5, 1e300, ints, 1 << 31) == 0
    assert c.seen[0] == (t.data_ptr(), -5, None, -(1 << 40), 0.5, 1e300, ctypes.addressof(ints), -(1 << 31))
    c.rc = 7
    assert c.launch(12345, True, c_void_p(777), 1, 2, 3, t[1:], 0) == 7
    assert c.seen[1] == (12345, 1, 777, 1, 2.0, 3.0, t.data_ptr() + 4, 0)


def test_many_arguments_on_the_stack():
    kinds = "pqif" * 8 + "pq" * 10
    c = Calls(kinds)
    args = [i + 1 if k != "f" else i + 0.25 for i, k in enumerate(kinds)]
    assert c.launch(*args) == 0 and list(c.seen[0]) == args


def test_whole_numbers_of_other_kinds():
    """What says which whole number it is stands for it, as with ctypes; what is none is refused."""
    c = Calls("iq")
    c.launch(np.int64(-3), np.uint8(200))
    c.launch(torch.tensor(4), np.int32(5))
    assert c.seen == [(-3, 200), (4, 5)]
    for bad in (1.0, np.float32(2.0), "3", None, torch.tensor(1.5)):
        with pytest.raises(TypeError):
            c.launch(bad, 0)
        with pytest.raises(TypeError):
            c.launch(0, bad)
    assert len(c.seen) == 2


@pytest.mark.parametrize("bad", [np.zeros(3, dtype=np.float32), np.float32(1.0), np.int64(5), b"bytes", bytearray(8), memoryview(b"x"), 1.5, "text",
                                 object(), [1]])
def test_what_is_no_pointer(bad):
    c = Calls("pi")
    with pytest.raises(TypeError):
        c.launch(bad, 1)
    assert not c.seen


def test_wrong_numbers_of_arguments_and_signatures():
    c = Calls("pi")
    for args in ((), (None,), (None, 1, 2)):
        with pytest.raises(TypeError):
            c.launch(*args)
    with pytest.raises(TypeError):
        c.launch(None, x=1)
    launch = build.load_extension("host_call").Launch
    for kinds in ("z", "i" * 45, "f" * 9):
        with pytest.raises(ValueError):
            launch(1, kinds)
    with pytest.raises(ValueError):
        launch(0, "i")


def test_recorded_launches_again():
    """The first addresses of the bound tensors are replaced wherever they stand as pointers, and nothing else is."""
    a, b = Calls("pipp", True), Calls("pqp", False)
    scratch, old, new = torch.zeros(8), (torch.zeros(2, 3), None, torch.zeros(5)), (torch.ones(2, 3), None, torch.ones(5))
    with record() as r:
        a.launch(old[0], old[0].data_ptr() & 0x7fffffff, scratch, 99)
        a.launch(scratch, 3, old[2], 99)
        b.launch(old[0], 1, 99)                                # not recorded
        a.rc = 801
        a.launch(old[0], 4, None, 99)                          # refused by its library: not made again
        a.rc = 0
    a.launch(old[0], 5, None, 99)                              # after the end
    assert r.bind(old) is True
    a.seen.clear(), b.seen.clear()
    assert r.run(new) == 0 and not b.seen
    assert a.seen == [(new[0].data_ptr(), old[0].data_ptr() & 0x7fffffff, scratch.data_ptr(), 99), (scratch.data_ptr(), 3, new[2].data_ptr(), 99)]
    assert r.run(old) == 0 and a.seen[2][0] == old[0].data_ptr()


def test_tensors_that_do_not_fit_a_place():
    a = Calls("pi", True)
    flat = torch.zeros(64)
    old = torch.zeros(16)
    assert old.data_ptr() % 16 == 0 and flat.data_ptr() % 16 == 0
    with record() as r:
        a.launch(old, 1)
    assert r.bind((old, None))
    a.seen.clear()
    for bad in (torch.zeros(17), torch.zeros(4, 4), torch.zeros(16, dtype=torch.int32), flat[1:17], torch.zeros(32)[::2], None, "x"):
        assert r.run((bad, None)) is None
    assert r.run((flat[4:20], flat)) is None                   # a tensor where there was none
    with pytest.raises(TypeError):
        r.run((old,))
    assert not a.seen and r.run((flat[4:20], None)) == 0 and a.seen == [(flat.data_ptr() + 16, 1)]


def test_what_does_not_bind():
    a = Calls("pipp", True)
    t, u = torch.zeros(4), torch.zeros(4)
    with record() as r:
        a.launch(t, 1, u, 99)
    assert r.bind((t, u)) is True and r.bind((t, t)) is False and r.bind((t, torch.zeros(4, 4).t()[1:])) is False
    with record() as r:
        a.launch(t, 1, u.data_ptr() + 4, 99)                   # an address as a number: inside one of the tensors, or not
    assert r.bind((t, u)) is False
    with record() as r:
        a.launch(t, 1, 0, 99)                                  # no address; the last one is the stream
    assert r.bind((t, u)) is True


def test_one_record_a_thread():
    with record():
        with pytest.raises(RuntimeError):
            with record():
                pass
    with record() as r:
        pass
    assert r.bind(()) is True and r.run(()) == 0


class Layer:
    """What `AlikeLayers` asks of a block: three launches, the second of which may fail."""

    def __init__(self, calls):
        self.calls, self.w, self.forwards = calls, torch.zeros(4), 0

    def alike(self, ctx, entry, writes_cache):
        return ("layer",), (self.w,)

    def first_norm(self):
        return None

    def forward(self, h, ctx, entry, writes_cache):
        self.forwards += 1
        for i, c in enumerate(self.calls):
            ops._check(c.launch(self.w, i, h, 99), "launch")
        return h


class After:
    def alike(self):
        return ("norm",), ()


class Ctx:
    norm_ahead, norm_after_block = None, After()


def test_a_recorded_launch_that_fails_ends_the_step(monkeypatch):
    from minfer_amd.engine.alike import AlikeLayers
    calls = [Calls("pipp", True) for _ in range(3)]
    monkeypatch.setattr(ops, "_trace", None)
    layers, run, h = [Layer(calls) for _ in range(4)], AlikeLayers(), torch.zeros(4)
    for layer in layers[:2]:
        assert run.forward(layer, h, Ctx(), 0, True) is h
    assert [l.forwards for l in layers] == [1, 0, 0, 0]
    assert [c.seen[1] for c in calls] == [(layers[1].w.data_ptr(), i, h.data_ptr(), 99) for i in range(3)]
    calls[1].rc = 719
    with pytest.raises(ops.KernelError):
        run.forward(layers[2], h, Ctx(), 0, True)
    assert [len(c.seen) for c in calls] == [3, 3, 2]           # nothing behind the one that failed


def test_a_layer_with_an_address_inside_a_tensor_runs_by_itself():
    from minfer_amd.engine.alike import AlikeLayers

    class Inside(Layer):
        def forward(self, h, ctx, entry, writes_cache):
            self.forwards += 1
            self.calls[0].launch(self.w.data_ptr() + 4, 0, h, 99)
            return h
    calls = [Calls("pipp", True)]
    layers, run, h = [Inside(calls) for _ in range(3)], AlikeLayers(), torch.zeros(4)
    for layer in layers:
        run.forward(layer, h, Ctx(), 0, True)
    assert [l.forwards for l in layers] == [1, 1, 1]
    assert [s[0] for s in calls[0].seen] == [l.w.data_ptr() + 4 for l in layers]
