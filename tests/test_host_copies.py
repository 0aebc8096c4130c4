"""Values on their way to and from the device: the ring of pinned slots uploads go through, the polled pieces of a read."""
import os
import subprocess
import sys

import numpy as np
import pytest


# the ring's slots are used again and again: every upload reads what the host wrote last, at each size and remainder
@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 3, 5, 64, 1023, 4097, 16384])
def test_a_slot_of_the_ring_is_read_anew(hip, n):
    for again in range(4):
        sent = [np.arange(n, dtype=np.uint32) * np.uint32(2654435761) + np.uint32(again * 100 + i) for i in range(20)]
        held = [hip.ndarray_from_vec_u32(a, [n]) for a in sent]
        for a, t in zip(sent, held):
            assert np.array_equal(hip.to_vec(t), a)


# ---- on the CPU: the same copies over a stand-in runtime (fake_hip.cpp), which can refuse a launch --------------------

FAKE = """
import ctypes, importlib, sys, time
import numpy as np
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
cg = importlib.import_module("catgrad-rs_amd")
be = cg.Backend(cg.load_library(), flags=int(sys.argv[2]))
a = np.arange(2000, dtype=np.uint32)

def refuse(kernel, n=1):
    fake.fake_hip_refuse(kernel.encode(), n)

def fails(f):
    t0, waits = time.time(), fake.fake_hip_waits()
    try:
        f()
    except cg.BackendPanic:
        assert fake.fake_hip_waits() > waits, "launches may still be storing into the buffers"
        assert time.time() - t0 < 0.2, f"found out by running out of time: {time.time() - t0:.3f} s"
        return True
    return False

def works():
    for i in range(20):     # more than there are slots, each read back at once, then all of them
        assert np.array_equal(be.to_vec(be.tensor(a + np.uint32(i))), a + np.uint32(i))
    held = [be.tensor(a * np.uint32(i)) for i in range(20)]
    for i, t in enumerate(held):
        assert np.array_equal(be.to_vec(t), a * np.uint32(i))
    big = np.arange(40 * 32768 + 7, dtype=np.uint32)    # more than both halves of the buffer reads go through
    assert np.array_equal(be.to_vec(be.tensor(big)), big)
    t0 = time.time()
    be.sync()
    assert time.time() - t0 < 0.2

works()
"""


@pytest.fixture(scope="module")
def fake_hip(tmp_path_factory):
    here, rocm = os.path.dirname(os.path.abspath(__file__)), os.environ.get("ROCM_PATH", "/opt/rocm")
    so = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(rocm, "include"), "-I" + os.path.join(os.path.dirname(here), "catgrad-rs_amd", "csrc"),
                           os.path.join(here, "fake_hip.cpp"), "-o", so])

    def run(script, flags=0):
        root = os.path.dirname(here)
        env = dict(os.environ, PYTHONPATH=root)
        p = subprocess.run([sys.executable, "-c", FAKE + script, so, str(flags)], cwd=root, env=env, capture_output=True, text=True, timeout=100)
        assert p.returncode == 0, p.stdout[-1000:] + p.stderr[-2000:]
    return run


EAGER = 2


@pytest.mark.parametrize("flags", [0, EAGER])
def test_copies_over_the_stand_in(fake_hip, flags):
    fake_hip("", flags)


def test_an_upload_that_was_not_launched_gives_its_slot_back(fake_hip):
    """The launch is refused on the queue's thread: the next wait reports it at once, and every slot can be used again."""
    fake_hip("""
refuse("from_host_kernel")
t = be.tensor(a)
assert fails(lambda: be.to_vec(t))
works()
refuse("from_host_kernel", 5)      # ... among others, with nothing read before the ring comes round
assert fails(lambda: [be.tensor(a + np.uint32(i)) for i in range(20)] and be.sync())
works()
""")


@pytest.mark.parametrize("words,flags", [(2000, 0), (3 * 32768, 0), (40 * 32768, 0), (2000, EAGER), (40 * 32768, EAGER)])
def test_a_read_that_was_not_launched_is_reported_at_once(fake_hip, words, flags):
    for n in (1, 2, 3) if words > 32 * 32768 else (1,):   # the first, second or third launch of the read
        fake_hip(f"""
big = np.arange({words}, dtype=np.uint32)
t = be.tensor(big)
be.sync()
refuse("to_host_kernel", {n})
assert fails(lambda: be.to_vec(t))
assert np.array_equal(be.to_vec(t), big)
works()
""", flags)


def test_a_prefetch_or_wait_that_was_not_launched(fake_hip):
    fake_hip("""
t = be.tensor(a[:500])
be.sync()
refuse("to_host_kernel")
be.prefetch(t)
assert fails(lambda: be.to_vec(t))
assert np.array_equal(be.to_vec(t), a[:500])
refuse("to_host_kernel")
assert fails(be.sync)
be.sync()
refuse("to_host_kernel")           # refused, and its tensor given up unread: the buffer is used again
t = be.tensor(a[:500])
be.prefetch(t)
del t
fails(be.sync)
for i in range(40):
    t = be.prefetch(be.tensor(a[:500] + np.uint32(i)))
    assert np.array_equal(be.to_vec(t), a[:500] + np.uint32(i))
works()
""")


def test_results_of_one_launch_cross_the_bus_together(fake_hip):
    """max(softmax(x)) and argmax(x): one copy for both, each by itself for many rows; a copy that was not launched, and one given up unread."""
    fake_hip("""
lang, nn = cg.lang, cg.nn
fake.fake_hip_launched.restype = ctypes.c_char_p

class Best(lang.Module):
    def path(self): return lang.path(["best"])
    def sort(self): return [lang.TENSOR], [lang.TENSOR] * 2
    def def_(self, b, args): return [lang.max(b, nn.softmax(b, args[0])), lang.argmax(b, args[0])]

it = cg.Interpreter(be, cg.stdlib())
term = Best().term()
run = lambda rows: it.run(term, [be.tensor(np.zeros((rows, 8), np.float32))])

def copies(reads):
    be.sync()
    fake.fake_hip_launched()
    for t in reads: be.to_vec(t)
    return fake.fake_hip_launched().decode().count("to_host_kernel")

for rows, n in ((5, 1), (8192, 1), (8193, 2)):
    p, k = run(rows)
    c = copies([p, k]), copies([p, k])
    assert c == ((1, 0) if n == 1 else (2, 2)), (rows, c)
    p, k = run(rows)
    be.realize(p)       # (asked for first, the column is found by itself)
    assert copies([k, p, k]) == (1 if n == 1 else 3), rows
del p, k
held = [run(5) for i in range(20)]      # more than there are buffers
c = [copies(r) for r in held]
assert c == [1] * 16 + [2] * 4, c
del held
p, k = run(5)
be.realize(p)
be.sync()
refuse("to_host_kernel")
assert fails(lambda: be.to_vec(p))
assert copies([p, k]) == 1
for i in range(40):
    p, k = run(5)
    be.realize(p)
    assert copies([k]) == 1
works()
""")


def test_a_kept_copy_is_not_read_once_something_was_launched(fake_hip):
    """Between the reads of two results that crossed together: a launch, which may have flagged an error, and copies to the host, which cannot."""
    fake_hip("""
lang, nn = cg.lang, cg.nn
fake.fake_hip_launched.restype = ctypes.c_char_p

class Best(lang.Module):
    def path(self): return lang.path(["best"])
    def sort(self): return [lang.TENSOR], [lang.TENSOR] * 2
    def def_(self, b, args): return [lang.max(b, nn.softmax(b, args[0])), lang.argmax(b, args[0])]

it = cg.Interpreter(be, cg.stdlib())
term = Best().term()
other, third = be.tensor(a[:64]), be.tensor(a[64:128])
be.realize(other), be.realize(third)

def copies(f):
    fake.fake_hip_launched()
    f()
    return fake.fake_hip_launched().decode().count("to_host_kernel")

for again in range(40):     # (more often than there are buffers)
    p, k = it.run(term, [be.tensor(np.zeros((5, 8), np.float32))])
    assert copies(lambda: be.to_vec(p)) == 1
    assert copies(lambda: be.to_vec(k)) == 0
    be.to_vec(other), be.prefetch(third), be.sync()
    assert copies(lambda: be.to_vec(k)) == 0
    be.realize(be.add(other, third))
    assert copies(lambda: be.to_vec(k)) == 1
    be.realize(be.add(other, third))
    assert copies(lambda: (be.to_vec(p), be.to_vec(k))) == 1
    assert copies(lambda: (be.to_vec(p), be.to_vec(k))) == 0
works()
""")


def test_results_are_read_one_by_one_without_room_for_them_on_the_host(fake_hip):
    fake_hip("""
lang, nn = cg.lang, cg.nn

class Best(lang.Module):
    def path(self): return lang.path(["best"])
    def sort(self): return [lang.TENSOR], [lang.TENSOR] * 2
    def def_(self, b, args): return [lang.max(b, nn.softmax(b, args[0])), lang.argmax(b, args[0])]

p, k = cg.Interpreter(be, cg.stdlib()).run(Best().term(), [be.tensor(np.zeros((5, 8), np.float32))])
be.realize(p)
be.sync()
refuse("hipHostMalloc")
assert not fails(lambda: be.to_vec(p)) and not fails(lambda: be.to_vec(k))
works()
""")
