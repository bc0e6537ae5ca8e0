"""The library's device memory and downloads (og_runtime.c) on the CPU, with
host stand-ins for the HIP calls (hip_stub.c): which device a block is
allocated on, what is kept and given back, and what is left of the calling
thread's device and pending error."""
import ctypes as C
import os
import subprocess
import threading

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
MB = 1 << 20
CAP = MB          # a 64th of the stand-in's 64 MB


@pytest.fixture()
def lib(tmp_path):
    so = str(tmp_path / "stub.so")
    subprocess.run(["gcc", "-O1", "-g", "-std=gnu11", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", "-I" + os.path.join(ROOT, "opengraph_amd", "csrc"),
                    "-I" + os.path.join(ROOT, "include"), os.path.join(HERE, "hip_stub.c"), "-o", so, "-lpthread",
                    "-Wl,-Bsymbolic"], check=True, timeout=120)
    x = C.CDLL(so)   # (bound inside: a HIP runtime loaded in the process is not called)
    x.og_dalloc.restype = C.c_void_p
    x.og_dalloc.argtypes = [C.c_size_t]
    x.og_dfree.argtypes = [C.c_void_p]
    for f in (x.stub_device_of, x.stub_size_of):
        f.argtypes = [C.c_void_p]
    x.stub_size_of.restype = x.stub_used.restype = C.c_size_t
    x.stub_limit.argtypes = [C.c_size_t]
    x.og_download.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t]
    assert x.ogpu_init(1) == 0
    return x


def test_blocks_are_the_librarys_devices(lib):
    """... whatever device the calling thread has chosen, which it keeps."""
    got = []

    def run():
        lib.stub_set(0, 0)      # a thread of its own starts on device 0
        a = lib.og_dalloc(5000)
        got.append((lib.stub_device_of(a), lib.stub_current()))
        lib.og_dfree(a)

    t = threading.Thread(target=run)
    t.start()
    t.join()
    assert got == [(1, 0)]
    b = lib.og_dalloc(5000)     # the same block, handed to this thread
    assert lib.stub_device_of(b) == 1


def test_kept_memory_is_bounded_and_given_back(lib):
    p = [lib.og_dalloc(300_000) for _ in range(10)]
    for x in p:
        lib.og_dfree(x)
    assert 0 < lib.stub_used() <= CAP
    lib.og_dfree(lib.og_dalloc(2 * MB))      # larger than all that is kept: never kept
    assert lib.stub_used() <= CAP
    live = lib.og_dalloc(300_000)
    assert lib.ogpu_release_memory() == 0
    assert lib.stub_used() == lib.stub_size_of(live)
    lib.og_dfree(live)


def test_an_allocation_fails_only_without_kept_memory(lib):
    for x in [lib.og_dalloc(300_000) for _ in range(3)]:
        lib.og_dfree(x)
    lib.stub_limit(950_001)
    a = lib.og_dalloc(950_001)               # not the rounded size, and nothing else
    assert lib.stub_size_of(a) == 950_001 == lib.stub_used()
    assert lib.og_dalloc(1) is None
    assert lib.stub_last() == 0              # reported, not left for another call to find
    lib.og_dfree(a)
    assert lib.og_dalloc(1)


@pytest.mark.parametrize("known", [0, 1])
@pytest.mark.parametrize("words", [1, MB - 1, MB, 9 * MB // 4 + 3])
def test_download_leaves_the_threads_state(lib, known, words):
    """Data whole, the thread's device and its pending error as they were."""
    lib.stub_known(known)
    src = (C.c_uint32 * words)(*([0] * 7)) if words >= 7 else (C.c_uint32 * words)()
    for i in range(0, words, 4099):
        src[i] = i * 2654435761 % (1 << 32)
    src[words - 1] = 77
    for device, error in ((0, 0), (1, 0), (0, 1), (1, 719)):
        dst = (C.c_uint32 * words)()
        lib.stub_set(device, error)
        assert lib.og_download(dst, src, words * 4) == 0
        assert (lib.stub_current(), lib.stub_last()) == (device, error)
        assert bytes(dst) == bytes(src)
