"""Conductance terms that a programmed matrix keeps between reads, ordered between streams.

The noisy MFMA read samples a program's conductance terms once where they do not depend on the
read event (memfast/reference.py:36-46) and later reads load them.  They are written on the
stream of the read that samples them; a read on another stream waits for that work first.
Everything else a read writes is its own call's.
"""

import threading

import torch

from . import hip


class _Written:
    """Work queued on one stream that other streams' reads wait for."""

    def __init__(self, device):
        self._event = torch.cuda.Event()
        self.record(device)

    def record(self, device):
        self.stream = hip._stream(device).value
        self._event.record(torch.cuda.current_stream(device))
        self._done = False

    def order(self, tensor):
        """Order the current stream's next work, which reads ``tensor``, after this; whether
        that is another stream.  The allocator then keeps ``tensor``'s memory for it."""
        device = tensor.device
        other = hip._stream(device).value != self.stream
        if not self._done:
            if self._event.query():
                self._done = True
            elif other:
                torch.cuda.current_stream(device).wait_event(self._event)
        if other:
            tensor.record_stream(torch.cuda.current_stream(device))
        return other


class KeptTerms:
    """A matrix's kept terms (``buffer``), what they were sampled from (``source``) and the
    lock under which a read takes them and queues its kernels, so that two threads' kernels
    do not interleave.  A copy of the matrix starts without any of it."""

    def __init__(self):
        self.lock = threading.RLock()
        self.buffer = self.source = self._written = self._built = None
        self._shared = False     # streams other than the writing one have read the buffer

    def __deepcopy__(self, memo):
        return type(self)()

    def __reduce__(self):
        return type(self), ()

    def take(self, size, device, source):
        """(buffer of at least ``size`` bytes, whether it holds the terms of ``source``: the
        same codes object, version and seed).  Without them the next read samples into it:
        ``queued`` follows once that read is queued.  Terms that other streams may still be
        reading are left to them."""
        held, buffer = self.source, self.buffer
        fits = buffer is not None and buffer.numel() >= size and buffer.device == device
        if fits and held is not None and held[0] is source[0] and held[1:] == source[1:]:
            self._shared = self._written.order(buffer) or self._shared
            return buffer, True
        self.source = None
        if not fits or self._shared or (self._written is not None and
                                        self._written.stream != hip._stream(device).value):
            self.buffer = buffer = torch.empty(max(1, size), dtype=torch.uint8, device=device)
            self._written, self._shared = None, False
        return buffer, False

    def queued(self, source):
        """The read that samples the terms of ``source`` into the buffer is queued."""
        device = self.buffer.device
        if self._written is None:
            self._written = _Written(device)
        else:
            self._written.record(device)
        self.source = source

    def built(self, codes):
        """The kernels' copy ``codes`` was made on the current stream."""
        self._built = codes, _Written(codes.device)

    def order_codes(self, codes):
        """Order the current stream after the work that made ``codes`` (``built``)."""
        if self._built is not None and self._built[0] is codes:
            self._built[1].order(codes)


__all__ = ["KeptTerms"]
