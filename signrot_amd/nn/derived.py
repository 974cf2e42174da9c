"""Tensors derived from a module's weight buffers once and kept beside them
(a rearranged copy for a kernel that reads another layout)."""
import weakref

import torch


class _Kept:
    """A derived value with the tensors it was made from (weakly, so that a
    buffer that is replaced is freed), their state, and the event after which
    it is written, until that was seen to have passed.  A copy of the module
    (deepcopy, pickle) starts without one."""

    def __init__(self, sources=(), state=None, value=None, event=None):
        self.refs = tuple(weakref.ref(t) for t in sources)
        self.state, self.value, self.event = state, value, event

    def __reduce__(self):
        return (_Kept, ())

    def holds(self, sources, state):
        return (len(self.refs) == len(sources) and self.state == state
                and all(r() is t for r, t in zip(self.refs, sources)))


def derived(module, name, sources, make):
    """make(*sources), kept on the module as `name` until one of the source
    tensors is replaced, moved or changed in place (by its version counter: a
    write through .data is not seen).

    The copy is launched on the first caller's stream; a caller on another one
    waits for it there.  Inside a graph capture a missing copy is recorded
    into the graph and not kept, since nothing has been written when the
    capture ends; a kept one is ordered before the capture by the capture's
    own synchronization.  Tensors without version counters (made under
    inference_mode) get a copy per call."""
    try:
        state = tuple((t.data_ptr(), t._version) for t in sources)
    except RuntimeError:
        return make(*sources)
    capturing = torch.cuda.is_current_stream_capturing()
    kept = module.__dict__.get(name)
    if kept is None or not kept.holds(sources, state):
        value = make(*sources)
        if not capturing:
            event = torch.cuda.Event()
            event.record(torch.cuda.current_stream(sources[0].device))
            module.__dict__[name] = _Kept(sources, state, value, event)
        return value
    event = kept.event
    if event is not None and not capturing:
        if event.query():
            kept.event = None
        else:
            torch.cuda.current_stream(sources[0].device).wait_event(event)
    return kept.value
