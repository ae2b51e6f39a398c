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


def test_q4k_plan_does_not_depend_on_scratch():
    """a Q4_K call captured without scratch takes the tile plan of the expanded call (and is accepted
    wherever its own plan was: no split-K workspace that only the other plan would need)"""
    run("""
def fc():
    out = []
    for k, n, g in launches():
        if k.startswith("k_gemm_fc") or k == "k_gemv_fc":
            out.append((k, re.findall(r"L[a-z]+([0-9]+)E", n)[:-1], g))      # all but the weight form
    return out

for M in (700, 1023, 1024, 1025, 2056, 4097):
    for N, K in ((100, 256), (768, 768), (1024, 1024), (2304, 768), (3072, 768), (4096, 512)):
        for f, x in ((c.gemm_dq_f32in, X), (c.gemm_dq, X)):
            if f == c.gemm_dq_f32in and M * N >= 4096 * 3072:
                continue                       # the rounding pass needs scratch of its own
            fresh = ema.Context(0)
            g = getattr(fresh, f.__name__)
            fresh.graph_begin()
            g(12, W, N, K, x, M, B, 1, R, Y)
            fresh.graph_end().destroy()
            captured = fc()
            g(12, W, N, K, x, M, B, 1, R, Y)
            eager = fc()
            fresh.close()
            assert captured and captured == eager, (M, N, K, captured, eager)
""")


def test_q4k_expands_where_it_measured_faster():
    """both sides of the rule's lines, fp32 and fp16 rows (times beside the rule)"""
    run("""
rule = [  # M, N, expanded with fp32 rows, with fp16 rows
    (699, 768, 0, 0), (700, 768, 1, 1), (700, 1024, 1, 1), (4112, 768, 1, 1), (4097, 1536, 1, 1),
    (1285, 1536, 0, 0), (1542, 1536, 1, 0), (2056, 1536, 1, 1), (1023, 2304, 0, 0), (1023, 4096, 0, 0), (1025, 2304, 1, 0), (1285, 2304, 1, 0),
    (1542, 2304, 1, 1), (1024, 3072, 1, 0), (1025, 3072, 1, 1), (1285, 4096, 0, 1), (1542, 4096, 0, 1),
    (2056, 4096, 1, 1)]
for M, N, f32, f16 in rule:
    c.gemm_dq_f32in(12, W, N, 768, X, M, B, 0, None, Y)
    assert ("k_expand_q4" in kernels()) == bool(f32), (M, N, "fp32 rows")
    c.gemm_dq_y16(12, W, N, 768, X, M, B, 0, None, Y)
    assert ("k_expand_q4" in kernels()) == bool(f16), (M, N, "fp16 rows")
    c.gemm_dq_f32in(8, W, N, 768, X, M, B, 0, None, Y)
    assert "k_expand_q4" not in kernels()
""")


def test_conv_split_k_follows_the_kernel():
    """256 workgroups of at least 18 slabs of 16 k for the convolutions on three bf16 parts (one
    workgroup per CU); 512 of at least 9 for the other packed ones, IC % 32 != 0 or 2 GiB images"""
    run("""
for side, ic, oc, ksz in ((64, 48, 128, 3), (16, 48, 512, 3), (32, 80, 128, 3), (16, 240, 512, 3), (64, 144, 256, 3), (64, 128, 128, 3),
                          (64, 256, 256, 3), (16, 512, 512, 3), (32, 96, 40, 3), (32, 128, 3, 3), (8, 16, 24, 5)):
    c.conv2d_ex(X, side, side, ic, 1, None, W, ksz, ksz, oc, 1, ksz // 2, None, None, Y)
    (k, _, grid), *reduce = launches()
    wide = oc > 16 and ic % 32 == 0
    assert k == ("k_conv2d_split" if wide else "k_conv2d_pkn" if oc <= 16 else "k_conv2d_pk"), k
    target, least = (256, 18) if wide else (512, 9)
    bm, bn = (256, 16) if oc <= 16 else (128, 128)
    tiles, slabs = -(-side * side // bm) * -(-oc // bn), ic * ksz * ksz // 16
    want = min(-(-target // tiles), slabs // least)
    per = slabs if tiles >= target * 3 // 4 or want < 2 else -(-slabs // want)
    per += per % 2 if wide else 0
    assert grid[2] == -(-slabs // per), (side, ic, oc, grid, per)
    assert [r[0] for r in reduce] == (["k_conv_reduce"] if grid[2] > 1 else [])
""")


def test_attention_route():
    """the kernel by strides and length: whole head up to 272 keys, the long one beyond, whole head
    again up to 512 keys for rows closer together than a head, else the one for any strides"""
    run("""
def route(f, S, D=48, H=3, B=2, st=None, **kw):
    E = H * D
    f(X, X + 0x1000, X + 0x2000, st or (1, 3 * E, D, 3 * E * S), D, S, H, B, 0.1, Y, **kw)
    (k, n, grid), = launches()
    return (k, int(re.findall(r"L[a-z]+([0-9]+)E", n)[1])) if k == "k_attn_head" else k

close = lambda S: (1, 16, 16 * S + 48, 3 * (16 * S + 48))
f32, f16 = c.flash_attn_f16kv, lambda *a, **kw: c.flash_attn_f16in(*a, None, (1, 144, 48, 144 * a[5]), **kw)
for f in (f32, f16):
    assert [route(f, S) for S in (1, 64, 65, 128, 129, 272)] == [("k_attn_head", t) for t in (4, 4, 8, 8, 17, 17)]
    assert [route(f, S) for S in (273, 512)] == ["k_attn_long"] * 2
    assert [route(f, S, st=close(S)) for S in (272, 273, 384, 385, 512)] == [("k_attn_head", t) for t in (17, 24, 24, 32, 32)]
assert route(f32, 513) == route(f32, 70000) == "k_attn_long"
assert route(f32, 513, st=close(513)) == "k_flash_attn_f16kv"
assert route(f32, 600, st=(2, 300, 100, 300 * 600)) == route(f32, 20, st=(2, 300, 100, 6000)) == "k_flash_attn_f16kv"
# more threads than a launch of the long kernel may have
assert route(f16, 400, D=16, H=64, B=65535) == ("k_attn_head", 32)
assert route(f32, 600, D=16, H=64, B=65535) == "k_flash_attn_f16kv"
try:
    f16(X, X + 0x1000, X + 0x2000, (1, 432, 48, 432 * 513), 48, 513, 3, 2, 0.1, Y)
    raise SystemExit("no error")
except ema.MghError:
    pass
""")
