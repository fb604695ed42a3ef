"""Order of a layer's calls, whose scratch is shared, on a model of torch's streams: which streams the stream of a call is
made to wait for, eagerly and while streams are capturing.  Runs on the CPU: the streams are objects that note what is
asked of them, and a wait that would tie an eager stream to a capture, or a capture to work ahead of it, fails at once.
"""
import contextlib
from types import SimpleNamespace

import pytest

from tilexr_amd import layer


class Stream:
    """`capture`: the running capture the stream belongs to, None while it is eager."""

    def __init__(self, name, handle, stream_id=None):
        self.name, self.cuda_stream = name, handle
        self.stream_id = handle + 100 if stream_id is None else stream_id
        self.capture, self.behind = None, set()

    def wait_stream(self, other):
        if self.capture is None and self.name == "own":
            self.capture = other.capture        # the layer's own stream, forked for a call on a wrapped one
        elif self.capture is None:
            assert other.capture is None, f"eager {self.name} is pulled into the capture of {other.name}"
        else:
            assert other.capture == self.capture, f"the capture of {self.name} waits for {other.name}, which is not in it"
        self.behind |= {other.name} | other.behind

    def __eq__(self, other):
        return isinstance(other, Stream) and self is other

    def __ne__(self, other):
        # as torch's: anything that is no stream, None among it, is neither equal nor unequal to one
        return isinstance(other, Stream) and self is not other

    __hash__ = object.__hash__

    def __repr__(self):
        return self.name


class Device:
    def __init__(self, monkeypatch):
        self.current = Stream("start", 1)
        self.own = Stream("own", 2)
        cuda = SimpleNamespace(current_stream=lambda device=None: self.current, stream=self.use,
                               is_current_stream_capturing=lambda: self.current.capture is not None)
        monkeypatch.setattr(layer.torch, "cuda", cuda)
        self.calls = layer._CallStream("cuda:0", self.own)

    @contextlib.contextmanager
    def use(self, stream):
        before, self.current = self.current, stream
        try:
            yield
        finally:
            self.current = before

    def call(self, stream):
        with self.use(stream), self.calls as (handle, current):
            assert current is stream
            return handle


@pytest.fixture
def device(monkeypatch):
    return Device(monkeypatch)


def test_eager_calls_wait_for_the_previous_stream_only_where_it_is_another(device):
    a, b = Stream("a", 10), Stream("b", 11)
    assert device.call(a) == 10 and device.call(a) == 10 and not a.behind - {"own"}
    device.call(b)
    assert "a" in b.behind
    device.call(a)
    assert "b" in a.behind


def test_eager_call_after_a_captured_one_waits_for_the_last_eager_one(device):
    a, b, c = Stream("a", 10), Stream("b", 11), Stream("c", 12)
    device.call(a)
    b.capture = 1
    device.call(b)
    b.capture = None
    device.call(c)
    assert "a" in c.behind


def test_eager_call_on_the_stream_that_captured_waits_for_the_last_eager_one(device):
    a, b = Stream("a", 10), Stream("b", 11)
    device.call(a)
    b.capture = 1
    device.call(b)
    b.capture = None
    device.call(b)
    assert "a" in b.behind


def test_eager_call_beside_a_running_capture_stays_out_of_it(device):
    a, b, c = Stream("a", 10), Stream("b", 11), Stream("c", 12)
    device.call(a)
    b.capture = 1
    device.call(b)
    device.call(c)
    assert "a" in c.behind and "b" not in c.behind
    # nor where the last eager stream is the one that is capturing now
    c.capture = 2
    device.call(a)
    assert "c" not in a.behind


def test_capture_is_not_ordered_behind_what_ran_before_it(device):
    a, b = Stream("a", 10), Stream("b", 11)
    device.call(a)
    b.capture = 1
    device.call(b)
    assert "a" not in b.behind


@pytest.mark.parametrize("eager_first", [None, "main", "side"])
def test_calls_of_one_capture_are_ordered_on_whatever_branch(device, eager_first):
    main, side, third = Stream("main", 10), Stream("side", 11), Stream("third", 12)
    if eager_first is not None:
        device.call({"main": main, "side": side}[eager_first])
    for s in (main, side, third):
        s.capture = 1
    device.call(main)
    device.call(side)
    assert "main" in side.behind
    device.call(third)
    assert "side" in third.behind
    device.call(main)
    assert "third" in main.behind


def test_calls_of_one_capture_are_ordered_around_an_eager_one(device):
    main, side, beside = Stream("main", 10), Stream("side", 11), Stream("beside", 12)
    device.call(main)
    main.capture = side.capture = 1
    device.call(main)
    device.call(beside)
    device.call(side)
    assert "main" in side.behind


def test_next_capture_does_not_wait_for_the_streams_of_the_one_before(device):
    a, b = Stream("a", 10), Stream("b", 11)
    a.capture = 1
    device.call(a)
    a.capture = None
    b.capture = 2
    device.call(b)
    assert "a" not in b.behind


def test_wrapped_streams_of_a_capture_share_the_layers_own(device):
    wrapped, b = Stream("wrapped", 10, stream_id=10), Stream("b", 11)
    wrapped.capture = b.capture = 1
    assert device.call(wrapped) == device.own.cuda_stream
    device.call(b)
    assert {"own", "wrapped"} <= b.behind and "own" in wrapped.behind
