"""Host-side pieces of the native library, compiled for the host alone: no GPU needed."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "pmpic_amd", "csrc")
HIPCC = os.environ.get("HIPCC") or shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.fixture(scope="module")
def checks(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("host") / "checks.so")
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-std=c++17", "-O1", "-fPIC", "-shared",
                    "-I", CSRC, os.path.join(HERE, "host", "checks.hip"), "-o", out], check=True)
    return ctypes.CDLL(out)


@pytest.mark.parametrize("cell", [0, 1, 2**25 - 1, 2**25, 2**26 - 1])
@pytest.mark.parametrize("head", [0, 17, 63])
def test_packed_runs_hold_every_cell_of_a_slot_table(checks, cell, head):
    """The binning packs a cell and a lane in 32 bits; grids with a slot table have up to 2^26
    cells, so the packed cell reaches the top bit."""
    out = (ctypes.c_int32 * 2)()
    checks.host_run_round_trip(cell, head, out)
    assert tuple(out) == (cell, head)


MB = 1 << 20


def _copy(checks, host, dev, bytes_each, parts, to_host, pinned, device=1):
    """(status, error left pending, blocks of pinned memory taken, copy commands, the calling
    thread's device afterwards, waits for the stream, bytes of the largest command) of a copy of a
    context on device 1."""
    out = (ctypes.c_int * 7)()
    checks.host_copy(ctypes.c_void_p(host.ctypes.data), ctypes.c_void_p(dev.ctypes.data),
                     ctypes.c_int64(bytes_each), parts, int(to_host), pinned, device, out)
    return list(out)


@pytest.mark.parametrize("bytes_each,parts,to_host,threads",
                         [(3 * MB + 17, 1, True, 1), (5 * MB - 3, 4, True, 4)])
@pytest.mark.parametrize("pinned", [0, 1, 2, 4])
def test_host_copies_without_pinned_memory(checks, bytes_each, parts, to_host, threads, pinned):
    """Copies of a size that goes through pinned slots, one thread's or four's, while the system gives
    pinned memory to some or none of the threads: every byte arrives, the copy reports success and
    leaves no error for the caller's next check to find."""
    rng = np.random.default_rng(bytes_each + pinned)
    src = rng.integers(0, 256, bytes_each * parts, dtype=np.uint8)
    dst = np.zeros_like(src)
    host, dev = (dst, src) if to_host else (src, dst)
    out = _copy(checks, host, dev, bytes_each, parts, to_host, pinned)
    assert out[:2] == [0, 0]
    np.testing.assert_array_equal(dst, src)
    assert out[2] == min(pinned, threads)
    assert out[3] == (parts if pinned == 0 else parts * -(-bytes_each // MB))


@pytest.mark.parametrize("bytes_each,parts,to_host,threads",
                         [(MB - 1, 1, True, 0), (MB, 1, True, 1), (16 * MB - 1, 1, True, 1),
                          (16 * MB, 1, True, 4), (MB // 4 - 8, 17, True, 0), (MB // 4, 17, True, 1),
                          (MB // 2, 7, True, 0), (MB // 2, 8, True, 1), (3 * MB // 4 - 8, 2, True, 0),
                          (3 * MB // 4, 2, True, 1), (MB, 17, True, 4), (MB, 1, False, 0), (40 * MB, 1, False, 0),
                          (2 * MB, 17, False, 0)])
def test_host_copies_route(checks, bytes_each, parts, to_host, threads):
    """Which copies go through pinned slots: to the host from 1 MB in parts of 768 KB or more, from 4 MB
    in parts of 256 KB or more, by four threads from 16 MB; from the host, where the runtime is as fast or faster, none."""
    src = np.arange(bytes_each * parts, dtype=np.uint8)
    dst = np.zeros_like(src)
    host, dev = (dst, src) if to_host else (src, dst)
    out = _copy(checks, host, dev, bytes_each, parts, to_host, 4)
    assert out[:3] == [0, 0, threads]
    np.testing.assert_array_equal(dst, src)


@pytest.mark.parametrize("to_host", [False, True])
@pytest.mark.parametrize("size", [1000, 3 * MB, 40 * MB])
@pytest.mark.parametrize("device", [0, 1])
def test_host_copies_leave_the_current_device(checks, size, to_host, device):
    """A copy of a context on device 1 by a thread whose current device is another: it succeeds (its
    events are made on the context's device) and the thread's device is what it was."""
    src = np.arange(size, dtype=np.uint8)
    dst = np.zeros_like(src)
    host, dev = (dst, src) if to_host else (src, dst)
    out = _copy(checks, host, dev, size, 1, to_host, 4, device)
    assert out[:2] == [0, 0] and out[4] == device
    np.testing.assert_array_equal(dst, src)


@pytest.mark.parametrize("to_host", [False, True])
def test_small_host_copies_wait_for_nothing(checks, to_host):
    """A copy through the runtime leaves the wait for the stream to the caller: parcel fields taken one
    after another wait once, not once a field."""
    src = np.arange(15_360, dtype=np.uint8)
    dst = np.zeros_like(src)
    host, dev = (dst, src) if to_host else (src, dst)
    out = _copy(checks, host, dev, len(src), 1, to_host, 4)
    assert out == [0, 0, 0, 1, 1, 0, len(src)]
    np.testing.assert_array_equal(dst, src)


@pytest.mark.parametrize("size,pieces", [(1, 1), (MB - 1, 1), (MB, 2), (1_024_000 + MB - 1, 2),
                                         (1_024_000 + MB, 3), (20 * MB, 21)])
def test_uploads_come_in_pieces(checks, size, pieces):
    """Uploads stay below the megabyte from which the runtime pins the caller's pages."""
    src = np.random.default_rng(size).integers(0, 256, size, dtype=np.uint8)
    dst = np.zeros_like(src)
    out = _copy(checks, src, dst, size, 1, False, 4)
    assert out[:3] == [0, 0, 0] and out[3] == pieces and out[6] < MB
    np.testing.assert_array_equal(dst, src)
