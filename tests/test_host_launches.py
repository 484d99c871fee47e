"""The host side of libgsq.so on a stand-in for the HIP runtime (hip_host_stub.cpp): which launches
and allocations a call makes. Runs in a child process, where libgsq.so binds to the stand-in."""
import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(os.path.dirname(HERE), "mlx-gsq-rco_amd", "mlx_gsq_amd", "libgsq.so")

PRELUDE = """
import ctypes, sys, threading
stub = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)
lib = ctypes.CDLL(sys.argv[2])
stub.stub_malloc_bytes.restype = ctypes.c_size_t
stub.stub_launch_kernel.restype = ctypes.c_void_p
I, P, F = ctypes.c_int64, ctypes.c_void_p, ctypes.c_float
for fn in (lib.gsq_qmm, lib.gsq_qmm_noalloc, lib.gsq_qmv):
    fn.argtypes = [ctypes.c_int, P, P, ctypes.c_int, P, ctypes.c_int, I, I, I, P]
lib.gsq_prepare.argtypes = [P]
lib.gsq_last_error.restype = ctypes.c_char_p
F32, F16, BF16 = 0, 1, 2
Q4_K, X, PACKED, Y, S = 12, 1 << 20, 1 << 24, 1 << 28, 1 << 32

def knob(name, value, kind=ctypes.c_int):
    kind.in_dll(stub, name).value = value

def call(fn, xdt=F16, m=200, n=1536, k=5120, x=X, stream=S):
    rc = fn(Q4_K, PACKED, x, xdt, Y, F32, m, n, k, stream)
    assert rc == 0, lib.gsq_last_error()

def counted(fn, *a, **kw):
    n = stub.stub_launches()
    call(fn, *a, **kw)
    return stub.stub_launches() - n
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no g++")
    so = str(tmp_path_factory.mktemp("stub") / "hip_host_stub.so")
    subprocess.run([cxx, "-std=c++17", "-O1", "-shared", "-fPIC", "-pthread", "-o", so,
                    os.path.join(HERE, "hip_host_stub.cpp")], check=True)
    return so


def run(stub, body):
    r = subprocess.run([sys.executable, "-c", PRELUDE + body, stub, LIB], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


def test_launches_of_one_call_stay_together(stub):
    """Calls that pass data through a stream's workspace (or the allocation-free entry point's scratch)
    in several launches: another thread's call on that stream never lands between them."""
    run(stub, """
lib.gsq_prepare(S)
# split tiles, summed by a second launch; bf16 and unaligned fp16 rows, laid out by a launch before;
# an unaligned matrix-vector row, copied by one; and the allocation-free entry point
CALLS = [(lib.gsq_qmm, {}), (lib.gsq_qmm, dict(xdt=BF16)), (lib.gsq_qmm, dict(x=X + 2, m=20)),
         (lib.gsq_qmv, dict(x=X + 2, m=1)), (lib.gsq_qmm_noalloc, {}), (lib.gsq_qmm_noalloc, dict(n=1000))]
lens = [counted(fn, **kw) for fn, kw in CALLS]
assert lens == [2, 3, 2, 2, 2, 2], lens
stub.stub_clear()
knob("stub_launch_us", 100)
def work(i):
    stub.stub_thread(i)
    for _ in range(20):
        call(CALLS[i][0], **CALLS[i][1])
threads = [threading.Thread(target=work, args=(i,)) for i in range(len(CALLS))]
[t.start() for t in threads]
[t.join() for t in threads]
log = [stub.stub_launch_thread(i) for i in range(stub.stub_launches())]
assert len(log) == 20 * sum(lens)
for group in ({0, 1, 2, 3}, {4, 5}):  # the workspace's users; the scratch's
    seq = [t for t in log if t in group]
    i = 0
    while i < len(seq):
        n = lens[seq[i]]
        assert seq[i:i + n] == [seq[i]] * n, f"call of thread {seq[i]} interrupted: {seq[i:i + n]}"
        i += n
""")


def test_staging_area_is_made_when_needed(stub):
    """The 128 MB in which fp32, bf16 and unaligned activations are laid out: not for callers of aligned
    fp16 rows, asked for again after a failure, never under capture, and by gsq_prepare_staging."""
    run(stub, """
MB = 1 << 20
lib.gsq_prepare_staging.argtypes = [P]
def big():
    return [b // MB for b in map(stub.stub_malloc_bytes, range(stub.stub_mallocs())) if b >= MB]
lib.gsq_prepare(S)
call(lib.gsq_qmm)
call(lib.gsq_qmv, x=X + 2, m=1)  # its copy uses the partials' memory
assert big() == [128], big()  # the partial tiles
# no room: the generic kernel; the next call asks again
knob("stub_malloc_limit", MB, ctypes.c_size_t)
assert counted(lib.gsq_qmm, xdt=BF16) == 1
knob("stub_malloc_limit", 1 << 40, ctypes.c_size_t)
assert counted(lib.gsq_qmm, xdt=BF16) == 3
assert big() == [128, 128]
assert counted(lib.gsq_qmm, xdt=F32, m=20) == 2 and big() == [128, 128]
# a stream that captures: nothing is allocated; prepared for it, the staged kernels are captured
T, U = S + 1, S + 2
assert lib.gsq_prepare(T) == 0 and lib.gsq_prepare_staging(U) == 0
assert big() == [128] * 5
knob("stub_capturing", 1)
assert counted(lib.gsq_qmm, xdt=BF16, stream=T) == 1
assert counted(lib.gsq_qmm, xdt=BF16, stream=U) == 3
assert lib.gsq_prepare_staging(T) != 0 and b"before the stream starts capturing" in lib.gsq_last_error()
assert big() == [128] * 5
knob("stub_capturing", 0)
knob("stub_malloc_limit", MB, ctypes.c_size_t)
assert lib.gsq_prepare_staging(T) != 0 and b"staging" in lib.gsq_last_error()
""")


def test_launch_attributes_per_device(stub):
    """A kernel's dynamic LDS limit is raised on every device it is launched on, and asked for again
    after a failure."""
    run(stub, """
lib.gsq_attn_seq.argtypes = [P, I, P, I, P, I, P, P, P, P, P, P, P, I, P, I, I, I, I, I, I, I, F, ctypes.c_int, P]
lib.gsq_attn_decode.argtypes = [P, I, P, I, P, I, P, P, P, P, P, P, P, I, I, I, I, I, I, I, F, P, I, ctypes.c_int, P]
lib.gsq_qmv_group2.argtypes = [ctypes.c_int, P, I, P, ctypes.c_int, P, I, P, P, ctypes.c_int, I, P]

def attn_seq(S_):
    return lib.gsq_attn_seq(X, 1024, X, 128, X, 128, X, X, X, X, X, X, Y, 512, X, 1, 64, 4, 1, 128, 64, 128, 1e-6, F16, S_)

def attn_decode(S_):
    return lib.gsq_attn_decode(X, 1024, X, 128, X, 128, X, X, X, X, X, X, Y, 512, 1, 4, 1, 128, 64, 128, 1e-6, None, 0, F16, S_)

def product(fn, m):
    return lambda S_: fn(Q4_K, PACKED, X, F16, Y, F32, m, 17408, 5120, S_)

def group(S_):
    return lib.gsq_qmv_group2(Q4_K, PACKED, 17408, Y, Q4_K, PACKED, 17408, Y + (1 << 20), X, F32, 5120, S_)

# prompt and single-token attention; the vector, quad-row and shared matrix-vector kernels; the
# small-batch and the tiled product
for i, fn in enumerate((attn_seq, attn_decode, product(lib.gsq_qmv, 1), product(lib.gsq_qmv, 4), group,
                        product(lib.gsq_qmm, 40), product(lib.gsq_qmm, 512))):
    knob("stub_device", 0)
    lib.gsq_prepare(S + i)
    stub.stub_clear()
    knob("stub_attr_fails", 1)
    assert fn(S + i) != 0, i
    assert stub.stub_launches() == 0, i
    knob("stub_attr_fails", 0)
    for device in (0, 1, 1, 0, 70, 70):
        knob("stub_device", device)
        assert fn(S + i) == 0, (i, lib.gsq_last_error())
    got = [stub.stub_attr_device(j) for j in range(stub.stub_attrs())]
    assert got == [0, 1, 70, 70], (i, got)  # past the 64 devices that are remembered: every time
""")
