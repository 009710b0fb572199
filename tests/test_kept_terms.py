"""Order between streams of the conductance terms a matrix keeps (memfast_amd/kept.py), on the
CPU with recorded streams and events."""

import copy

import pytest
import torch

from memfast_amd import hip, kept


class FakeStream:
    def __init__(self, handle):
        self.handle, self.waited = handle, []

    def wait_event(self, event):
        self.waited.append(event)


class FakeEvent:
    def __init__(self):
        self.recorded, self.done = [], False

    def record(self, stream):
        self.recorded.append(stream)
        self.done = False

    def query(self):
        return self.done


@pytest.fixture
def device(monkeypatch):
    """Streams 1, 2, .. by handle; ``use`` makes one current.  Uses of memory by streams other
    than its own are listed in ``used``."""
    streams, state = {}, dict(current=1)

    def current(_=None):
        return streams.setdefault(state["current"], FakeStream(state["current"]))

    class Device:
        used = []
        stream = staticmethod(current)

        @staticmethod
        def use(handle):
            state["current"] = handle

    class Pointer:
        value = property(lambda self: state["current"])

    monkeypatch.setattr(hip, "_stream", lambda device: Pointer())
    monkeypatch.setattr(torch.cuda, "Event", FakeEvent)
    monkeypatch.setattr(torch.cuda, "current_stream", current)
    monkeypatch.setattr(torch.Tensor, "record_stream",
                        lambda tensor, stream: Device.used.append((tensor.data_ptr(), stream.handle)))
    return Device


CPU = torch.device("cpu")


def sampled(terms, codes, seed=1):
    """(buffer, whether it held the terms) of a read, which samples them otherwise."""
    source = (codes, codes._version, seed)
    held = terms.held(CPU, source)
    if held is not None:
        return held, True
    buffer = terms.fresh(64, CPU)
    terms.queued(source, waits=False)
    return buffer, False


def test_another_stream_waits_for_the_samples(device):
    terms, codes = kept.KeptTerms(), torch.zeros(4)
    first, reuse = sampled(terms, codes)
    assert not reuse
    event = terms._written._event
    again, reuse = sampled(terms, codes)
    assert reuse and again is first and not device.stream().waited and not device.used
    device.use(2)
    other, reuse = sampled(terms, codes)
    assert reuse and other is first and device.stream().waited == [event]
    assert device.used == [(first.data_ptr(), 2)]
    event.done = True
    device.use(3)
    sampled(terms, codes)
    assert not device.stream().waited and (first.data_ptr(), 3) in device.used
    del device.used[:]


def test_new_samples_leave_terms_in_use_alone(device):
    """Reprogrammed codes are sampled in place on the stream that wrote the terms, and into
    memory of their own once another stream has read them or writes them."""
    terms, codes = kept.KeptTerms(), torch.zeros(4)
    first, _ = sampled(terms, codes)
    codes.add_(1)
    second, reuse = sampled(terms, codes)
    assert not reuse and second is first
    device.use(2)
    sampled(terms, codes)
    device.use(1)
    codes.add_(1)
    third, reuse = sampled(terms, codes)
    assert not reuse and third.data_ptr() != first.data_ptr()
    device.use(2)
    fourth, reuse = sampled(terms, torch.zeros(4))
    assert not reuse and fourth is not third
    del device.used[:]


def test_terms_are_not_held_until_their_read_is_queued(device):
    terms, codes = kept.KeptTerms(), torch.zeros(4)
    source = (codes, codes._version, 1)
    assert terms.held(CPU, source) is None
    buffer = terms.fresh(64, CPU)      # (the read that follows raises)
    assert terms.held(CPU, source) is None and terms.fresh(64, CPU) is buffer
    terms.queued(source, waits=False)
    assert terms.held(CPU, source) is buffer
    assert terms.held(CPU, (codes, codes._version, 2)) is None
    assert terms.held(torch.device("meta"), source) is None


def test_a_read_that_its_call_waits_for_is_recorded_only_in_between(device):
    terms, codes = kept.KeptTerms(), torch.zeros(4)
    source = (codes, codes._version, 1)
    first = terms.fresh(64, CPU)
    number = terms.queued(source, waits=True)
    writer = device.stream()
    assert terms._written._event is None
    device.use(2)                      # another thread's read, before the call has waited
    assert terms.held(CPU, source) is first
    event = terms._written._event
    assert event.recorded == [writer] and device.stream().waited == [event]
    terms.settled(number)
    device.use(3)
    assert terms.held(CPU, source) is first and not device.stream().waited
    device.use(1)
    codes.add_(1)
    source = (codes, codes._version, 1)
    terms.fresh(64, CPU)
    later = terms.queued(source, waits=True)
    assert later != number
    terms.settled(number)              # (the earlier call again)
    device.use(4)
    terms.held(CPU, source)
    assert len(device.stream().waited) == 1
    terms.settled(later)
    del device.used[:]


def test_codes_built_on_one_stream_are_waited_for_on_another(device):
    terms, codes = kept.KeptTerms(), torch.zeros(4)
    terms.built(codes)
    device.use(2)
    terms.order_codes(torch.zeros(4))
    assert not device.stream().waited
    terms.order_codes(codes)
    assert len(device.stream().waited) == 1 and device.used == [(codes.data_ptr(), 2)]
    del device.used[:]


def test_a_copy_starts_without_terms(device):
    terms, codes = kept.KeptTerms(), torch.zeros(4)
    sampled(terms, codes)
    clone = copy.deepcopy(terms)
    assert clone.source is None and clone.buffer is None and clone.lock is not terms.lock
