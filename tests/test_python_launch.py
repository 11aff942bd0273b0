"""The Python side of a launch (tessera_amd/host/pylaunch.cpp): what arrives at the C entry point.  The entry here
is a callback, so no device and no library call is needed."""
import ctypes
import os
import subprocess
import sys
import sysconfig

import numpy as np
import pytest

from tessera_amd import KernelLaunch, backend as backend_module

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ENTRY = ctypes.CFUNCTYPE(ctypes.c_int32, ctypes.c_size_t, ctypes.POINTER(ctypes.c_uint32), ctypes.POINTER(ctypes.c_uint32),
                         ctypes.POINTER(ctypes.c_void_p), ctypes.POINTER(ctypes.c_size_t), ctypes.c_size_t,
                         ctypes.POINTER(ctypes.c_uint64), ctypes.c_size_t, ctypes.c_void_p)
LAUNCHES = [backend_module._launch_arrays, backend_module._launch_ctypes]   # (the first is the extension's, see below)


class FakeBuffer:
    def __init__(self, handle, size, then=lambda: None):
        self.handle, self.size, self.then = handle, size, then

    def Handle(self):
        self.then()
        return self.handle

    def Size(self):
        return self.size


def arrived(launch, kernel, arguments, stream, status=0):
    """(status, what the entry got) of one launch."""
    got = {}

    @ENTRY
    def entry(kernel, grid, block, buffers, sizes, nbuffers, scalars, nscalars, stream):
        got.update(kernel=kernel, grid=grid[:3], block=block[:3], buffers=[b or 0 for b in buffers[:min(nbuffers, 16)]],
                   sizes=sizes[:min(nbuffers, 16)], scalars=scalars[:min(nscalars, 16)], counts=(nbuffers, nscalars), stream=stream or 0)
        return status
    return launch(ctypes.cast(entry, ctypes.c_void_p).value, kernel, arguments, stream), got


@pytest.mark.parametrize("launch", LAUNCHES)
def test_arguments_arrive(launch):
    arguments = KernelLaunch(3, 2, 1, 64, 5, 7, [FakeBuffer(0x1000, 8), FakeBuffer(2 ** 47, 2 ** 40)],
                             [1, -1, 2 ** 64 + 5, np.uint64(9), np.int32(-2), True])
    status, got = arrived(launch, 11, arguments, 0x2000, status=4)
    assert status == 4
    assert got == {"kernel": 11, "grid": [3, 2, 1], "block": [64, 5, 7], "buffers": [0x1000, 2 ** 47], "sizes": [8, 2 ** 40],
                   "scalars": [1, 2 ** 64 - 1, 5, 9, 2 ** 64 - 2, 1], "counts": (2, 6), "stream": 0x2000}


@pytest.mark.parametrize("launch", LAUNCHES)
def test_counts_past_the_limits_arrive_as_they_are(launch):
    arguments = KernelLaunch(buffers=[FakeBuffer(i, i) for i in range(19)], scalars=list(range(21)))
    _, got = arrived(launch, 1, arguments, 0)
    assert got["counts"] == (19, 21) and got["buffers"] == list(range(16)) and got["scalars"] == list(range(16))


@pytest.mark.parametrize("launch", LAUNCHES)
def test_lists_changed_while_they_are_read(launch):
    """Handle() runs Python code, which may shorten the launch's lists (as another thread may): the launch is the one
    that the lists held when it was read."""
    buffers, scalars = [], [1, 2, 3]
    buffers.extend([FakeBuffer(0x10, 1, lambda: (buffers.clear(), buffers.append(None))), FakeBuffer(0x20, 2), FakeBuffer(0x30, 3)])
    _, got = arrived(launch, 1, KernelLaunch(buffers=buffers, scalars=scalars), 0)
    assert got["buffers"] == [0x10, 0x20, 0x30] and got["sizes"] == [1, 2, 3]

    class Shortening:
        def __int__(self):
            scalars.clear()
            return 7
    scalars[:] = [Shortening(), 8, 9]
    _, got = arrived(launch, 1, KernelLaunch(buffers=[], scalars=scalars), 0)
    assert got["scalars"] == [7, 8, 9] and scalars == []


@pytest.mark.parametrize("launch", LAUNCHES)
def test_errors_of_the_arguments_are_raised(launch):
    for bad in (KernelLaunch(buffers=[object()]), KernelLaunch(scalars=["x"]), KernelLaunch(scalars=5), KernelLaunch(grid_x=None)):
        with pytest.raises((AttributeError, ValueError, TypeError)):
            arrived(launch, 1, bad, 0)


def test_extension_is_built_for_this_interpreter():
    """Its file carries the interpreter's tag, so that no other loads it."""
    from tessera_amd import _native
    assert backend_module._launch_arrays is _native.launch
    assert _native.__file__.endswith(sysconfig.get_config_var("EXT_SUFFIX"))


def test_launches_without_the_extension():
    """An interpreter that the extension was not built for still launches, through ctypes."""
    program = ("import sys; sys.modules['tessera_amd._native'] = None\n"
               "import tessera_amd; from tessera_amd import backend as b\n"
               "assert b._launch_arrays is b._launch_ctypes\n"
               "be = tessera_amd.Backend(); k = be.LoadKernel('gemm_q4k')\n"
               "try:\n    be.LaunchKernel(k, tessera_amd.KernelLaunch(buffers=[be.WrapBuffer(0x1000, 1 << 20)] * 17, scalars=[1, 1, 256]))\n"
               "except tessera_amd.StatusError as e:\n    assert e.code == tessera_amd.StatusCode.InvalidArgument; print('refused')\n")
    out = subprocess.run([sys.executable, "-c", program], cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert out.stdout.strip() == "refused", out.stderr
