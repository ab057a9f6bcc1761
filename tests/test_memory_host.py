"""The library's device memory on the host: who gets a freed block, what the driver
is asked to do for it, and that nobody waits for another thread's driver call."""
import ctypes
import os
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

_HERE = os.path.dirname(os.path.abspath(__file__))
TEMP, KEPT, ANY = 0, 1, 2
NULL, SIDE, OTHER, PER_THREAD = 0, 0x1000, 0x2000, 2
UNUSED, ON_NULL, ELSEWHERE = 0, 1, 2
N = 100000
MB = 1 << 20
UNSUPPORTED = 3  # cr_status


class Memory:
    def __init__(self, path):
        self.lib = ctypes.CDLL(path)
        self.lib.mem_alloc.restype = ctypes.c_void_p
        self.lib.mem_alloc.argtypes = [ctypes.c_size_t, ctypes.c_int, ctypes.c_void_p]
        self.lib.mem_free.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
        self.lib.handle_free.argtypes = [ctypes.c_void_p, ctypes.c_uint]
        self.lib.set_capturing.argtypes = [ctypes.c_void_p, ctypes.c_int]
        self.lib.mem_sync.argtypes = [ctypes.c_void_p]
        self.lib.set_room.argtypes = [ctypes.c_size_t]
        self.lib.used.restype = ctypes.c_size_t
        self.lib.take_log.argtypes = [ctypes.c_char_p, ctypes.c_size_t]

    def alloc(self, use, s, n=N):
        return self.lib.mem_alloc(n, use, s)

    def log(self):
        b = ctypes.create_string_buffer(1 << 16)
        self.lib.take_log(b, len(b))
        return [x for x in b.value.decode().split(";") if x]

    # one call that uses `k` temporaries of a stream one after the other
    def call(self, s, k=1, n=N):
        self.lib.call_begin()
        got = []
        for _ in range(k):
            got.append(self.alloc(TEMP, s, n))
            self.lib.mem_free(got[-1], s)
        self.lib.call_end()
        return got


@pytest.fixture(scope="module")
def built(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("memory") / "memory_host.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-pthread", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", "-o", so, os.path.join(_HERE, "memory_host.cpp")], check=True)
    return so


@pytest.fixture
def mem(built, tmp_path):
    so = str(tmp_path / "memory.so")  # a copy: an empty cache
    with open(built, "rb") as f, open(so, "wb") as g:
        g.write(f.read())
    return Memory(so)


def test_temporaries_of_one_call(mem):
    a, b = mem.call(SIDE, 2)
    assert a == b
    assert mem.log() == ["malloc@%d" % SIDE, "sync@%d" % SIDE]
    assert mem.call(SIDE) == [a] and mem.call(OTHER) == [a]  # synchronised at the end of each call: anyone's


def test_null_stream_temporaries_need_no_synchronisation(mem):
    a, = mem.call(NULL)
    assert mem.call(NULL, 2) == [a, a]
    assert mem.log() == ["malloc@0"]
    assert mem.call(SIDE) != [a]  # another stream does not get it, and does not wait for it
    assert "sync@0" not in mem.log()


@pytest.mark.parametrize("stream", [NULL, SIDE])
def test_a_failed_call_leaves_nothing_pending(mem, stream):
    """Its grids and regridders may be destroyed next, and count as unused."""
    mem.lib.call_begin()
    mem.lib.mem_free(mem.alloc(TEMP, stream), stream)
    mem.lib.call_fail()
    mem.lib.call_end()
    assert mem.log()[-1] == "sync@%d" % stream


@pytest.mark.parametrize("stream", [PER_THREAD, SIDE])
def test_running_calls_keep_their_temporaries(mem, stream):
    """One stream handle on two threads (hipStreamPerThread: two streams)."""
    with ThreadPoolExecutor(1) as a, ThreadPoolExecutor(1) as b:
        a.submit(mem.lib.call_begin).result()
        b.submit(mem.lib.call_begin).result()
        p = a.submit(mem.alloc, TEMP, stream).result()
        a.submit(mem.lib.mem_free, p, stream).result()  # in order on a's stream; its work is pending
        q = b.submit(mem.alloc, TEMP, stream).result()
        assert q != p
        assert b.submit(mem.alloc, KEPT, stream).result() != p
        assert a.submit(mem.alloc, TEMP, stream).result() == p
        a.submit(mem.lib.mem_free, p, stream).result()
        mem.log()
        a.submit(mem.lib.call_end).result()
        assert mem.log() == ["sync@%d" % stream]
        assert b.submit(mem.alloc, TEMP, stream).result() == p
        b.submit(mem.lib.call_end).result()


@pytest.mark.parametrize("stream", [NULL, SIDE])
def test_what_a_call_has_freed_before_it_synchronises(mem, stream):
    with ThreadPoolExecutor(1) as other:
        mem.lib.call_begin()
        p, q = mem.alloc(TEMP, stream), mem.alloc(TEMP, stream, 9 * N)
        mem.lib.mem_free(p, stream)
        mem.lib.mem_sync(stream)
        mem.lib.mem_free(q, stream)
        assert other.submit(mem.alloc, ANY, OTHER).result() == p
        assert other.submit(mem.alloc, TEMP, OTHER, 9 * N).result() != q
        mem.log()
        mem.lib.call_end()
        assert mem.log() == (["sync@%d" % stream] if stream else [])


def test_handle_blocks_by_use(mem):
    def handle(bits):
        p = mem.alloc(KEPT, SIDE)
        mem.lib.handle_free(p, bits)
        mem.log()
        return p

    p = handle(UNUSED)  # no work pending
    assert mem.alloc(ANY, NULL) == p and mem.log() == []
    q = handle(ON_NULL)
    assert q != p and mem.alloc(TEMP, SIDE) not in (p, q)
    mem.log()
    assert mem.alloc(TEMP, NULL) == q and mem.log() == []
    r = handle(ON_NULL)
    assert mem.alloc(ANY, NULL) == r and mem.log() == ["sync@0"]
    for bits in (ELSEWHERE, ON_NULL | ELSEWHERE):
        t = handle(bits)
        assert mem.alloc(TEMP, SIDE) != t and mem.alloc(TEMP, NULL) != t
        assert "free" not in mem.log()  # temporaries do not wait for the device
        assert mem.alloc(KEPT, SIDE) == t
        assert mem.log() == ["malloc", "free"]  # hipFree waits for the device


def test_captures_are_left_alone(mem):
    """hipDeviceSynchronize breaks stream captures, on this and on other threads."""
    for bits in (UNUSED, ON_NULL, ELSEWHERE):
        for s in (NULL, SIDE, PER_THREAD):
            for use in (KEPT, ANY):
                mem.lib.handle_free(mem.alloc(use, s), bits)
            mem.call(s, 3)
    for i in range(400):
        mem.lib.handle_free(mem.alloc(KEPT, SIDE, 20000 + 4096 * (i % 90)), ELSEWHERE)
    log = mem.log()
    assert "devicesync" not in log and "malloc" in log and "free" in log
    assert not [x for x in log if "relaxed" in x]  # hipMalloc and hipFree otherwise break captures, too


@pytest.mark.parametrize("use", [TEMP, KEPT])
def test_capturing_streams_are_refused(mem, use):
    mem.call(SIDE)
    mem.log()
    mem.lib.set_capturing(SIDE, 1)
    mem.lib.call_begin()
    assert mem.alloc(use, SIDE) is None
    assert mem.alloc(use, NULL) is not None  # the null stream is not captured
    mem.lib.call_end()
    assert mem.log()[0] == "error%d" % UNSUPPORTED
    mem.lib.set_capturing(SIDE, 0)
    assert mem.alloc(use, SIDE) is not None


def test_no_lock_is_held_while_the_driver_works(mem):
    p = mem.alloc(ANY, NULL)
    mem.lib.handle_free(p, UNUSED)
    mem.lib.hold(1)
    with ThreadPoolExecutor(2) as ex:
        try:
            slow = ex.submit(mem.alloc, KEPT, SIDE, 50 * N)  # stops inside the driver
            assert mem.lib.wait_held()
            quick = ex.submit(lambda: (mem.alloc(ANY, NULL), mem.lib.handle_free(p, UNUSED)))
            assert quick.result(timeout=20)[0] == p
        finally:
            mem.lib.hold(0)
        assert slow.result(timeout=20)


@pytest.mark.parametrize("bits", [UNUSED, ON_NULL, ELSEWHERE])
def test_kept_memory_is_bounded(mem, bits):
    """1/64 of the device (1 MB here); past it a few larger trims, not one a free."""
    live = [mem.alloc(KEPT, SIDE, 30000 + 17000 * i) for i in range(24)]
    mem.log()
    for p in live:
        mem.lib.handle_free(p, bits)
    assert 0.5 * MB <= mem.lib.used() <= MB
    waits = mem.log().count("malloc")
    assert waits == (0 if bits != ELSEWHERE else waits) and waits <= 12


def test_temporaries_past_the_bound(mem):
    mem.lib.call_begin()
    p = [mem.alloc(TEMP, SIDE, MB) for _ in range(3)]
    for x in p:
        mem.lib.mem_free(x, SIDE)
    assert mem.lib.used() >= 3 * MB  # the running call may still want them
    mem.lib.call_end()
    assert mem.lib.used() <= MB
    assert mem.log()[3] == "sync@%d" % SIDE  # before anything goes back


def test_out_of_memory_gives_everything_back_first(mem):
    live = [mem.alloc(KEPT, SIDE, 3 * N) for _ in range(3)]
    for p, bits in zip(live, (UNUSED, ON_NULL, ELSEWHERE)):
        mem.lib.handle_free(p, bits)
    mem.lib.set_room(mem.lib.used() + N)
    assert mem.alloc(KEPT, SIDE, 8 * N) is not None
    mem.lib.set_room(mem.lib.used())
    assert mem.alloc(KEPT, SIDE, 8 * N) is None
