"""The host side of libmgh without a GPU: which kernels a call launches and what it does to the
context's buffers, on a recording HIP runtime (tests/fake_hip.cpp). Each case is a process of its own,
so that libmgh binds to that runtime."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
FAKE = os.path.join(ROOT, "tests", "_build", "libfake_hip.so")

PRELUDE = """
import ctypes, re, sys
sys.path.insert(0, %r)
fake = ctypes.CDLL(%r, mode=ctypes.RTLD_GLOBAL)
fake.fake_used.restype = ctypes.c_size_t
fake.fake_limit.argtypes = [ctypes.c_size_t]
import edge_maskgit_amd as ema
W, X, B, R, Y, G = (0x100000 * (i + 1) for i in range(6))       # addresses of operands, never read

def launches():
    '''[(kernel, template arguments and all, mangled, grid)] since the last call'''
    out = []
    for i in range(fake.fake_launches()):
        name, dims = ctypes.create_string_buffer(4096), (ctypes.c_uint * 6)()
        fake.fake_launch(i, name, 4096, dims)
        n = name.value.decode()
        out.append((re.search(r"k_[a-z0-9_]*[a-z0-9]", re.sub(r"([0-9])(k_)", r"\\1 \\2", n)).group(0), n, tuple(dims[:3])))
    fake.fake_clear()
    return out

def kernels():
    return [k for k, _, _ in launches()]

c = ema.Context(0)
""" % (ROOT, FAKE)


@pytest.fixture(scope="module", autouse=True)
def fake_hip():
    src = os.path.join(ROOT, "tests", "fake_hip.cpp")
    os.makedirs(os.path.dirname(FAKE), exist_ok=True)
    r = subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-I/opt/rocm/include", src, "-o", FAKE],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr


def run(body):
    r = subprocess.run([sys.executable, "-c", PRELUDE + body], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout


def test_scratch_survives_a_failed_growth():
    """a Q4_K call whose expanded weights find no memory decodes in the K loop in the scratch that
    is there, and later calls (captured ones too) still have it"""
    run("""
M, N, K = 4200, 3072, 768
c.gemm_dq_f32in(8, W, N, K, X, M, B, 0, None, Y)            # rounded activations in the scratch
assert "k_f32_to_f16" in kernels()
fake.fake_limit(fake.fake_used())                            # nothing more to be had
used = fake.fake_used()
c.gemm_dq_f32in(12, W, N, K, X, M, B, 0, None, Y)
k = kernels()
assert "k_expand_q4" not in k and "k_f32_to_f16" in k, k
assert fake.fake_used() == used
c.graph_begin()
c.gemm_dq_f32in(8, W, N, K, X, M, B, 0, None, Y)
c.gemm_dq_f32in(12, W, N, K, X, M, B, 0, None, Y)
c.graph_end().destroy()
try:
    c.gemm_dq_f32in(8, W, N, K, X, 2 * M, B, 0, None, Y)
    raise SystemExit("no error")
except ema.MghError as e:
    assert "out of memory" in str(e)
c.gemm_dq_f32in(8, W, N, K, X, M, B, 0, None, Y)             # the error is not another call's
# room for what the call needs but not for twice the old scratch
fake.fake_limit(used + (M * K * 2 + 255) // 256 * 256 + N * K * 2)
c.gemm_dq_f32in(12, W, N, K, X, M, B, 0, None, Y)
assert "k_expand_q4" in kernels()
c.close()
assert fake.fake_used() == 0
""")
