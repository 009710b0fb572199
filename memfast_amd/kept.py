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

    def __init__(self):
        self._event = self._queue = self.stream = None

    def queued(self, device):
        """The work is the newest on the current stream."""
        stream = hip._stream(device).value
        if self._queue is None or stream != self.stream:
            self.stream, self._queue = stream, torch.cuda.current_stream(device)
        self._recorded = self.done = False

    def record(self):
        """An event behind the work (and what its stream holds by now)."""
        if self._event is None:
            self._event = torch.cuda.Event()
        self._event.record(self._queue)
        self._recorded = True

    def order(self, tensor):
        """Order the current stream's next work, which reads ``tensor``, after this; whether
        that is another stream.  The allocator then keeps ``tensor``'s memory for it."""
        device = tensor.device
        if hip._stream(device).value == self.stream:
            return False
        current = torch.cuda.current_stream(device)
        if not self.done:
            if not self._recorded:
                self.record()
            self.done = self._event.query()
            if not self.done:
                current.wait_event(self._event)
        tensor.record_stream(current)
        return True


class KeptTerms:
    """A matrix's kept terms (``buffer``), what they were sampled from (``source``) and the
    lock under which a read takes them and queues its kernels, so that two threads' kernels
    do not interleave.  A copy of the matrix starts without any of it."""

    def __init__(self):
        self.lock = threading.RLock()
        self.buffer = self.source = self._written = self._built = None
        self._shared = False     # streams other than the writing one have read the buffer
        self._samples = 0        # reads that sampled

    def __deepcopy__(self, memo):
        return type(self)()

    def __reduce__(self):
        return type(self), ()

    def held(self, device, source):
        """The buffer, where it holds the terms of ``source`` on ``device`` (the same codes
        object, version and seed), ordered for the current stream; else None."""
        held, buffer = self.source, self.buffer
        if held is None or held[0] is not source[0] or held[1:] != source[1:]:
            return None
        if buffer.device != device:
            return None
        if self._written.order(buffer):
            self._shared = True
        return buffer

    def fresh(self, size, device):
        """A buffer of at least ``size`` bytes for new terms; ``queued`` follows once the read
        that samples them is queued.  Terms that other streams may still be reading are left
        to them."""
        buffer, written = self.buffer, self._written
        self.source = None
        if (buffer is None or buffer.numel() < size or buffer.device != device or self._shared
                or (written is not None and written.stream != hip._stream(device).value)):
            self.buffer = buffer = torch.empty(max(1, size), dtype=torch.uint8, device=device)
            self._written, self._shared = None, False
        return buffer

    def queued(self, source, waits):
        """The read that samples the terms of ``source`` into the buffer is queued; a number for
        ``settled``.  A read whose call ``waits`` for it needs no event unless another thread's
        read comes in between, and records it then; others record it now (a training step of
        784 -> 512 at 128 rows, which samples anew each time, 525 against 532 us)."""
        written = self._written
        if written is None:
            written = self._written = _Written()
        written.queued(self.buffer.device)
        if not waits:
            written.record()
        self.source = source
        self._samples += 1
        return self._samples

    def settled(self, number):
        """The call of read ``number`` has waited for it."""
        with self.lock:
            if self._written is not None and self._samples == number:
                self._written.done = True

    def built(self, codes):
        """The kernels' copy ``codes`` was made on the current stream."""
        written = _Written()
        written.queued(codes.device)
        written.record()
        self._built = codes, written

    def order_codes(self, codes):
        """Order the current stream after the work that made ``codes`` (``built``)."""
        if self._built is not None and self._built[0] is codes:
            self._built[1].order(codes)


__all__ = ["KeptTerms"]
