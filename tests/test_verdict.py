"""CPU tests of the bounds checks' host side: where a verdict is waited for, the words it is
written to, and which stores count as a call's own."""
import contextlib
import os
import shutil
import subprocess

import pytest
import torch

from tilemaxsim_amd import _lib
from tilemaxsim_amd.flash_pqsim_kernel import TileMaxSimPQ

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_words_of_an_earlier_check_are_not_taken_for_this_one(tmp_path):
    """tests/verdict_words.cpp against the polling code that the library uses."""
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "verdict_words")
    build = subprocess.run([gxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-I", os.path.join(REPO, "tilemaxsim_amd", "csrc"),
                            os.path.join(REPO, "tests", "verdict_words.cpp"), "-o", exe], capture_output=True, text=True)
    assert build.returncode == 0, build.stderr
    run = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0 and run.stdout == "ok\n", (run.returncode, run.stdout, run.stderr)


def test_codes_verdict_is_waited_for_on_the_codes_device(monkeypatch):
    """The check's launch, the scoring call and the verdict's wait all run with the codes'
    device current: a default stream handle names the current device's stream."""
    inside, calls = [], []

    @contextlib.contextmanager
    def on_device(dev):
        inside.append(dev)
        yield
        inside.pop()

    class Lib:
        def tms_codes_check(self, *args):
            calls.append(("check", list(inside)))
            return _lib.TMS_OK

        def tms_codes_verdict(self, verdict, stream):
            calls.append(("verdict", list(inside)))
            return _lib.TMS_OK

    monkeypatch.setattr(_lib, "load", Lib)
    monkeypatch.setattr(_lib, "on_device", on_device)
    monkeypatch.setattr(_lib, "stream_of", lambda t: 0)
    monkeypatch.setattr(_lib, "verdict_ptr", lambda: 64)
    pq = TileMaxSimPQ.__new__(TileMaxSimPQ)
    pq.K = 16
    codes = torch.zeros(4, dtype=torch.int32)

    def score():
        calls.append(("score", list(inside)))
        return "scores"

    assert pq._checked(codes, score) == "scores"
    assert calls == [(step, [codes.device]) for step in ("check", "score", "verdict")]
    # a scoring call that raises: its verdict is still read there, and the error is passed on
    calls.clear()

    def fails():
        raise MemoryError("no room for the scores")

    with pytest.raises(MemoryError):
        pq._checked(codes, fails)
    assert calls == [(step, [codes.device]) for step in ("check", "verdict")] and not inside


def test_verdict_words_do_not_follow_the_default_device(monkeypatch):
    """The words are host memory under any default device (pinning itself needs a GPU and is
    left out here; torch refuses to pin a tensor of another device)."""
    zeros = torch.zeros
    with torch.device("meta"):
        assert zeros(1).device.type == "meta"  # torch lists its constructors at first use, before the patch below

    def host_zeros(*args, pin_memory=False, **kw):
        words = zeros(*args, **kw)
        assert pin_memory and words.device.type == "cpu"
        return words

    monkeypatch.setattr(torch, "zeros", host_zeros)
    monkeypatch.delattr(_lib._thread, "verdict", raising=False)
    try:
        with torch.device("meta"):
            assert _lib.verdict_ptr() != 0
    finally:
        vars(_lib._thread).pop("verdict", None)  # made without pinning


def test_parts_are_a_thread_s_own_and_follow_its_stream(monkeypatch):
    """One buffer a thread, for the stream and device that it last used: calls of two threads,
    or on two streams, never share one."""
    import threading
    dev = torch.device("cpu")
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    vars(_lib._thread).pop("parts", None)
    first = _lib.parts_ptr(dev, 16)
    assert first != 0 and _lib.parts_ptr(dev, 16) == first
    held = _lib._thread.parts  # alive, so that its memory is not given out again
    seen = []

    def other():
        seen.append((_lib.parts_ptr(dev, 16), _lib._thread.parts))

    t = threading.Thread(target=other)
    t.start()
    t.join()
    assert seen[0][0] != first and _lib.parts_ptr(dev, 16) == first
    assert _lib.parts_ptr(dev, 32) != first and _lib._thread.parts is not held
    assert _lib.parts_ptr(torch.device("meta"), 32) == 0  # another device: its own buffer
    vars(_lib._thread).pop("parts", None)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    _lib.parts_ptr(dev, 48)  # under capture: nothing is kept
    assert not hasattr(_lib._thread, "parts")
