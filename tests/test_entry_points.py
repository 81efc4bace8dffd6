"""The table of bound entry points while another thread swaps the library
(``ezops.profiling.WaveTrace`` does): at every bytecode boundary of a lookup the
other thread swaps the library and looks an entry up (CPU, with stand-ins for
the two libraries)."""

import sys
from types import SimpleNamespace

from ezops import _hip


def _swapped_at(step: int, old, new):
    """``_fn("f")`` on `old`, interrupted before its `step`-th bytecode by a thread that
    swaps to `new` and looks ``g`` up.  -> (the looked-up entry, whether `step` was reached)"""
    seen = 0

    def tracer(frame, event, arg):
        nonlocal seen
        if frame.f_code is not _hip._fn.__code__:
            return None
        frame.f_trace_opcodes, frame.f_trace_lines = True, False
        if event == "opcode":
            if seen == step:
                sys.settrace(None)
                _hip._lib = new
                _hip._fn("g")
                sys.settrace(tracer)
            seen += 1
        return tracer

    sys.settrace(tracer)
    try:
        fn = _hip._fn("f")
    finally:
        sys.settrace(None)
    return fn, seen > step


def test_lookup_survives_a_library_swap_at_any_point(monkeypatch):
    monkeypatch.setattr(_hip, "_lib", None)
    for warm in (False, True):
        step, reached = 0, True
        while reached:
            old, new = SimpleNamespace(f="old f", g="old g"), SimpleNamespace(f="new f", g="new g")
            _hip._lib = old
            if warm:
                assert _hip._fn("g") == "old g"
            fn, reached = _swapped_at(step, old, new)
            assert fn in ("old f", "new f")  # whichever library the call met
            if reached:
                assert (_hip._fn("f"), _hip._fn("g")) == ("new f", "new g"), f"swap at step {step}"
                _hip._lib = old
                assert (_hip._fn("f"), _hip._fn("g")) == ("old f", "old g"), f"swap at step {step}"
            step += 1
        assert step > 20
