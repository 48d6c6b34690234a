"""What has to hold in the process while a HIP graph is recorded."""
from __future__ import annotations

import contextlib
import gc
import threading

_LOCK = threading.Lock()
_HOLDERS = 0
_RESUME = False


@contextlib.contextmanager
def collector_held():
    """Python's cyclic collector does not run by itself inside, in any thread. It comes whenever enough objects were made, and what
    it finds dead may be another captured graph (in a dropped worker, or in the frames that a kept exception holds): a graph
    that dies waits for the device, which is an error while a capture is under way, and an error out of a destructor ends
    the process. Holders may overlap; the last one out starts the collector again, if it ran before the first."""
    global _HOLDERS, _RESUME
    with _LOCK:
        if _HOLDERS == 0:
            _RESUME = gc.isenabled()
            gc.disable()
        _HOLDERS += 1
    try:
        yield
    finally:
        with _LOCK:
            _HOLDERS -= 1
            if _HOLDERS == 0 and _RESUME:
                gc.enable()
