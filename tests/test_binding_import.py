"""Importing the binding loads no torch (device memory and streams come from it only
once a call is made), and a call's default stream is torch's current one, with
torch's own error where there is no device to initialise."""
import os
import subprocess
import sys

import pytest

import kvhp

PKG = os.path.dirname(os.path.abspath(kvhp.__file__))


def test_import_loads_no_torch():
    code = f"import sys; sys.path.insert(0, {PKG!r}); import kvhp; assert 'torch' not in sys.modules"
    subprocess.run([sys.executable, "-c", code], check=True)


def test_default_stream_without_device():
    torch = pytest.importorskip("torch")
    if torch.cuda.is_available():
        pytest.skip("a device is there")
    with pytest.raises(Exception) as want:
        torch.cuda.current_stream()
    with pytest.raises(type(want.value)) as got:
        kvhp._stream(None)
    assert str(got.value) == str(want.value)


@pytest.mark.gpu
def test_default_stream_is_the_current_one():
    torch = pytest.importorskip("torch")
    code = (f"import sys; sys.path.insert(0, {PKG!r}); import kvhp, torch; "
            "assert not torch.cuda.is_initialized(); h = kvhp._stream(None); "
            "assert torch.cuda.is_initialized() and h == torch.cuda.current_stream().cuda_stream")
    subprocess.run([sys.executable, "-c", code], check=True)
    code = (f"import os, sys; sys.path.insert(0, {PKG!r}); import kvhp, torch; kvhp._stream(None)\n"
            "r, w = os.pipe()\n"
            "if os.fork() == 0:\n"
            "    try: kvhp._stream(None)\n"
            "    except RuntimeError as e: os.write(w, str(e).encode())\n"
            "    os._exit(0)\n"
            "os.close(w); os.wait(); sys.exit(0 if b'fork' in os.read(r, 4096) else 1)")
    subprocess.run([sys.executable, "-c", code], check=True)   # a forked child is refused
    side = torch.cuda.Stream()
    assert kvhp._stream(None) == torch.cuda.current_stream().cuda_stream
    with torch.cuda.stream(side):
        assert kvhp._stream(None) == side.cuda_stream
    assert kvhp._stream(side) == side.cuda_stream
